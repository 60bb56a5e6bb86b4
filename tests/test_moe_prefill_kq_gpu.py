"""The K-quant form of the prompt grouped expert product (moe_pf.hip,
moe_pf_kq_kernel: weights through registers a super-block ahead) at its edges:
one super-block and odd numbers of them, partial and single-row weight tiles,
runs around the 32- and 64-entry row tiles, and Q6_K weights at every byte
alignment."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from helpers import normalised_error
from oracle import qref
from swarmllm_amd._lib import X_BF16, X_F16
from test_moe_gpu import MOE_TYPES, expert_stack, t32
from test_moe_prefill_gpu import prefill_into

pytestmark = pytest.mark.gpu

RUNS = [1, 31, 32, 33, 0, 64, 65, 7]  # entries of each expert


def one_choice(seed):
    """Every token to one expert, the experts' runs of RUNS lengths."""
    n = sum(RUNS)
    ids = np.random.default_rng(seed).permutation(n).astype(np.int32)
    return ids, np.repeat(np.arange(len(RUNS)), RUNS).astype(np.int32), n


@pytest.mark.parametrize("name", ["Q4_K", "Q6_K"])
@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("n,k", [(1, 256), (129, 256), (128, 768), (200, 512)])
def test_edges(name, bf16, n, k):
    qtype = MOE_TYPES[name]
    ids, experts, tokens = one_choice(n + k)
    stack = expert_stack(qtype, len(RUNS), n, k, 5)
    x = np.random.default_rng(k).standard_normal((tokens, k)).astype(np.float32)
    rnd = qref.round_bf16 if bf16 else qref.round_f16
    xs = t32(x).to(torch.bfloat16 if bf16 else torch.float16)
    out = prefill_into(stack, xs, X_BF16 if bf16 else X_F16, k, ids, experts, None, 1, tokens)
    wb = stack.data_.cpu().numpy().reshape(len(RUNS), -1)
    for e in range(len(RUNS)):
        sel = ids[experts == e]
        if not len(sel):
            continue
        w = rnd(qref.to_float(qtype, wb[e], n * k).reshape(n, k)).astype(np.float64)
        xe = rnd(x[sel]).astype(np.float64)
        # exact products, k sums in f32: at most k 2^-24 of sum |w x| <=
        # ||w|| ||x||, and the result's own rounding
        assert normalised_error(out[sel], xe @ w.T, w, xe) <= (k + 1) * 2.0**-24


@pytest.mark.parametrize("shift", [1, 2, 3, 5, 13])
def test_q6_k_weights_at_any_byte(shift):
    qtype = MOE_TYPES["Q6_K"]
    n, k = 70, 768
    ids, experts, tokens = one_choice(3)
    stack = expert_stack(qtype, len(RUNS), n, k, 6)
    xs = t32(np.random.default_rng(4).standard_normal((tokens, k)).astype(np.float32)).half()
    want = prefill_into(stack, xs, X_F16, k, ids, experts, None, 1, tokens)
    data = stack.data_.reshape(-1)
    moved = torch.zeros(data.numel() + 64, dtype=torch.uint8, device=data.device)
    moved[shift:shift + data.numel()] = data.view(torch.uint8)
    other = SimpleNamespace(shape=stack.shape, dtype=stack.dtype, data_=moved[shift:])
    got = prefill_into(other, xs, X_F16, k, ids, experts, None, 1, tokens)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
