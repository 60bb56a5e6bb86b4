"""Q4_K at 1-2 rows of long weight rows: past the dispatch lines the multi-row
kernel takes the product (and at 2 rows the GLU gets a launch of its own), under them, and
without room for the activation's planes, the streaming kernel. Every product
keeps its bits: a weight row's result does not depend on how many rows its
weight has."""
import ctypes

import numpy as np
import pytest
import torch

from swarmllm_amd import GgmlDType, QMatMul, QTensor, forward_glu
from swarmllm_amd._lib import lib

pytestmark = pytest.mark.gpu


def weight(n, k, seed):
    rng = np.random.default_rng(seed)
    b = rng.integers(0, 256, (n * k // 256, 144), dtype=np.uint8)
    b[:, :4] = (rng.uniform(0.005, 0.02, (len(b), 2)).astype(np.float16)).view(np.uint8)
    return QTensor(torch.from_numpy(b.reshape(-1)).cuda(), (n, k), GgmlDType.Q4K)


def first(q, n):
    """The weight of q's first n rows."""
    k = q.shape[1]
    return QTensor(q.data_.reshape(-1)[:n * k // 256 * 144].clone(), (n, k), q.dtype)


def kernel():
    return lib().qmm_last_kernel().decode()


@pytest.mark.parametrize("rows,k,small,large", [(1, 8448, 4096, 4100), (1, 16384, 100, 4112), (2, 4352, 3072, 3073),
                                                 (2, 8192, 64, 3100)])
def test_forward_bits_across_the_line(rows, k, small, large):
    q = weight(large, k, k + rows)
    x = torch.randn(rows, k, device="cuda", generator=torch.Generator("cuda").manual_seed(rows))
    a = QMatMul(q).forward(x)
    assert "launch_nr(" in kernel()
    b = QMatMul(first(q, small)).forward(x)
    assert "launch_stream" in kernel()
    assert torch.equal(a[:, :small], b)


@pytest.mark.parametrize("rows,k,small,large", [(2, 4352, 1536, 1537), (2, 8192, 20, 1600)])
@pytest.mark.parametrize("act", ["silu", "gelu"])
def test_glu_bits_across_the_line(rows, k, small, large, act):
    g, u = weight(large, k, 1), weight(large, k, 2)
    x = 0.1 * torch.randn(rows, k, device="cuda", generator=torch.Generator("cuda").manual_seed(9))
    a = forward_glu(x, QMatMul(g), QMatMul(u), act)
    assert "launch_glu(" in kernel()
    b = forward_glu(x, QMatMul(first(g, small)), QMatMul(first(u, small)), act)
    assert "launch_glu_x" in kernel()
    assert torch.equal(a[:, :small], b)


def test_no_workspace_is_still_taken():
    """Products that quantize in their own launch need no workspace."""
    rows, k, n = 2, 4352, 8200
    g, u = weight(n, k, 3), weight(n, k, 4)
    x = 0.1 * torch.randn(rows, k, device="cuda", generator=torch.Generator("cuda").manual_seed(5))
    want = forward_glu(x, QMatMul(g), QMatMul(u), "silu")
    wg, wu = QMatMul(g).forward(x), QMatMul(u).forward(x)
    L, need = lib(), ctypes.c_size_t(0)
    out = torch.full((3, rows, n), float("nan"), device="cuda")
    ptrs = (ctypes.c_void_p * 2)(g.data_.data_ptr(), u.data_.data_ptr())
    dsts = (ctypes.c_void_p * 2)(out[0].data_ptr(), out[1].data_ptr())
    ns = (ctypes.c_int64 * 2)(n, n)
    st = torch.cuda.current_stream().cuda_stream
    assert L.qmm_forward_shared(int(g.dtype), 2, ptrs, ns, dsts, ns, x.data_ptr(), k, None, 0, ctypes.byref(need), k,
                                rows, 1, st) == 0
    assert L.qmm_forward_glu(int(g.dtype), 0, g.data_.data_ptr(), u.data_.data_ptr(), x.data_ptr(), k,
                             out[2].data_ptr(), n, None, 0, ctypes.byref(need), k, n, rows, 1, st) == 0
    torch.cuda.synchronize()
    assert torch.equal(out[0], wg) and torch.equal(out[1], wu) and torch.equal(out[2], want)
