"""The Q8_0 hidden-state wire codec on the device against the CPU oracle
(oracle/qref_wire.c, pinned in test_wire_oracle.py): encoded bytes and
decoded values bit for bit, at the sizes a layer split sends (a token's
hidden state of 4096 / 8192 values, a prompt chunk of 512 tokens) and at
lengths that leave a partial trailing group."""
import numpy as np
import pytest
import torch

from helpers import special_rows
from oracle import qref
from swarmllm_amd import quant
from swarmllm_amd._lib import QMM_UNSUPPORTED, lib

pytestmark = pytest.mark.gpu


def inputs(n: int, seed: int) -> np.ndarray:
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(n).astype(np.float32)
    ch = rng.permutation(n)[: max(1, n // 100)]
    x[ch] *= np.float32(20.0)
    return x


@pytest.mark.parametrize("n", [1, 31, 32, 33, 50, 4096, 8192, 512 * 4096, 4096 * 3 + 17])
def test_wire_encode_decode_bit_exact(n):
    x = inputs(n, n)
    xt = torch.from_numpy(x).cuda()
    b = quant.quantize_q8_0(xt)
    want = qref.wire_encode(x)
    assert b.numel() == want.size == quant.q8_0_byte_len_checked(n)
    assert np.array_equal(b.cpu().numpy(), want)
    y = quant.dequantize_q8_0(b, n).cpu().numpy()
    assert np.array_equal(y.view(np.uint32), qref.wire_decode(want, n).view(np.uint32))


def test_wire_special_values_bit_exact():
    """Zeros, ties of the rounding, subnormal-scale values, powers of two and
    non-finite values (skipped by the block maximum, coded by the clamp)."""
    sp = special_rows(96).ravel()
    extra = np.array([np.inf, -np.inf, np.nan, 2.5, -2.5, 127.0, 0.5, -0.5] + [1.0] * 24, np.float32)
    allbad = np.array([np.nan, np.inf, -np.inf] * 10 + [np.nan, np.nan], np.float32)
    x = np.concatenate([sp, extra, allbad, np.zeros(7, np.float32)]).astype(np.float32)
    b = quant.quantize_q8_0(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.array_equal(b, qref.wire_encode(x))
    y = quant.dequantize_q8_0(torch.from_numpy(b).cuda(), x.size).cpu().numpy()
    assert np.array_equal(y.view(np.uint32), qref.wire_decode(b, x.size).view(np.uint32))


def test_wire_rejects_a_wrong_length_and_takes_empty_input():
    with pytest.raises(ValueError):
        quant.dequantize_q8_0(torch.zeros(33, dtype=torch.uint8, device="cuda"), 32)
    st = lib().qmm_wire_decode(torch.zeros(68, dtype=torch.uint8, device="cuda").data_ptr(), 67, 50,
                               torch.empty(50, device="cuda").data_ptr(), 0)
    assert st == QMM_UNSUPPORTED
    assert quant.quantize_q8_0(torch.empty(0, device="cuda")).numel() == 0
    assert quant.dequantize_q8_0(torch.empty(0, dtype=torch.uint8, device="cuda"), 0).numel() == 0


@pytest.mark.parametrize("n", [7, 2047, 2048, 2049, 2056, 5 * 2048 + 40])
@pytest.mark.parametrize("xo,bo", [(0, 0), (1, 0), (0, 1), (3, 5), (4, 16)])
def test_wire_at_any_alignment_and_workgroup_edge(n, xo, bo):
    """Values and bytes at any offset from a 16-byte boundary (the vector
    accesses step aside) and lengths around a workgroup's 2048 values; nothing
    is written past the last byte or value."""
    x = inputs(n, n + xo)
    xb = torch.zeros(n + xo, device="cuda")
    xb[xo:] = torch.from_numpy(x).cuda()
    want = qref.wire_encode(x)
    nb = want.size
    out = torch.full((bo + nb + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    assert lib().qmm_wire_encode(xb.data_ptr() + 4 * xo, n, out.data_ptr() + bo, st) == 0
    got = out.cpu().numpy()
    assert np.array_equal(got[bo:bo + nb], want) and np.all(got[bo + nb:] == 0xA5) and np.all(got[:bo] == 0xA5)
    y = torch.full((xo + n + 16,), -7.0, device="cuda")
    assert lib().qmm_wire_decode(out.data_ptr() + bo, nb, n, y.data_ptr() + 4 * xo, st) == 0
    y = y.cpu().numpy()
    assert np.array_equal(y[xo:xo + n].view(np.uint32), qref.wire_decode(want, n).view(np.uint32))
    assert np.all(y[xo + n:] == -7.0) and np.all(y[:xo] == -7.0)
