"""The gate + up + GLU form of the single-pass Q4_K GEMM (one launch, neither
weight cut along K) gives, bit for bit, the two products followed by
the elementwise GLU: at its 256-row and 64-column tile edges, with odd n and a
padded output, for every activation."""
import ctypes

import pytest
import torch

from swarmllm_amd import GgmlDType, QMatMul, QTensor, _lib, fill_normal, forward_glu, glu
from swarmllm_amd._lib import lib
from swarmllm_amd.qtensor import quantize_act

pytestmark = pytest.mark.gpu


def pair(n, k, seed):
    return [QMatMul(QTensor.quantize(fill_normal(n * k, seed=seed + i, std=0.02).reshape(n, k), GgmlDType.Q4K))
            for i in range(2)]


@pytest.mark.parametrize("act", ["silu", "swiglu_oai", "gelu"])
@pytest.mark.parametrize("n,k,rows", [(14336, 2048, 512), (16385, 2048, 257), (33333, 2304, 129), (9000, 2048, 700)])
def test_one_launch_equals_the_composition(act, n, k, rows):
    gate, up = pair(n, k, n + k)
    x = fill_normal(rows * k, seed=rows).reshape(rows, k)
    print(f"n={n} k={k} rows={rows} {act}", flush=True)
    y = forward_glu(x, gate, up, act)
    assert "launch_gemm_q4k_sp_glu" in lib().qmm_last_kernel().decode()
    g, u = QMatMul.forward_shared(x, [gate, up])
    assert torch.equal(y, glu(g, u, act))


def test_weights_that_alone_would_be_cut_along_k():
    """1024 x 4096 at 512 rows: forward cuts such a weight, the gated form
    does not; its bits are the uncut products' (qmm_matmul)."""
    n, k, rows = 1024, 4096, 512
    mats = pair(n, k, 5)
    x = fill_normal(rows * k, seed=6).reshape(rows, k)
    y = forward_glu(x, *mats)
    assert "launch_gemm_q4k_sp_glu" in lib().qmm_last_kernel().decode()
    xq = quantize_act(x, _lib.ACT_Q8K)
    outs = []
    for m in mats:
        outs.append(torch.empty((rows, n), device="cuda"))
        assert lib().qmm_matmul(12, m.qtensor.data_.data_ptr(), xq.data_ptr(), outs[-1].data_ptr(), n, k, n, rows,
                                torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(y, glu(*outs))


def test_padded_output_rows_stay_untouched():
    n, k, rows, ldd = 20001, 2048, 300, 20010
    gate, up = pair(n, k, 7)
    x = fill_normal(rows * k, seed=8).reshape(rows, k)
    want = forward_glu(x, gate, up)
    out = torch.full((rows, ldd), float("nan"), device="cuda")
    need = ctypes.c_size_t(0)
    L = lib()
    assert L.qmm_forward_glu(12, 0, None, None, None, k, None, ldd, None, 0, ctypes.byref(need), k, n, rows, 0, 0) == 0
    ws = torch.empty(need.value, dtype=torch.uint8, device="cuda")
    assert L.qmm_forward_glu(12, 0, gate.qtensor.data_.data_ptr(), up.qtensor.data_.data_ptr(), x.data_ptr(), k,
                             out.data_ptr(), ldd, ws.data_ptr(), ws.numel(), ctypes.byref(need), k, n, rows, 1,
                             torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(out[:, :n], want) and bool(torch.isnan(out[:, n:]).all())
