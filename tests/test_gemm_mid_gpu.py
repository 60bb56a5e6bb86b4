"""Q4_K and Q6_K products of 17-128 rows (gemm_kq_mid.hip) against the CPU
oracle: at the edges of its row tiles (32, 64, 96), of its row chunks
(97, 129, 193 rows), of its 128-column tiles and of its K cut, and with the largest codes and
scales a block can hold; and the kernels that take such a product where the
workspace has no room for the slots of its cut.

Bound: the super-block sums are exact integers and the min sums exact f32, so
a result differs from the oracle's by f32 roundings only: per super-block
three (2^-24 each) of terms bounded by d dy sum |p y| + dmin dy sum |m S| and
one per addition, so at most (nsb + 4) 2^-24 of the sum of the terms'
magnitudes, which for these weights is below 3 ||w|| ||x||: 1.1e-5 at 56
super-blocks; 1e-5 is held (1e-7 measured)."""
import ctypes
import zlib

import numpy as np
import pytest
import torch

from helpers import normalised_error, special_rows, weights
from oracle import qref
from swarmllm_amd import GgmlDType, QMatMul, QTensor, _lib, fill_normal
from swarmllm_amd._lib import lib
from swarmllm_amd.qtensor import quantize_act

pytestmark = pytest.mark.gpu

BOUND = 1e-5
KERNEL = {qref.Q4_K: "launch_gemm_q4k_mid(", qref.Q6_K: "launch_gemm_q6k_mid("}


def no_slots_kernel(t, n, rows):
    """The kernel of a product that is cut, without room for its slots."""
    if t == qref.Q6_K and rows > 32:
        return "launch_gemm_q6k("
    few = -(-rows // 32) * -(-n // 4096) <= (3 if t == qref.Q6_K else 6)
    return ("launch_q6(" if t == qref.Q6_K else "launch_sk") if few else KERNEL[t]


SHAPES = [  # (n, k, rows)
    (129, 1536, 33), (1, 1536, 40), (128, 1792, 64), (300, 4096, 65), (2048, 2048, 96), (255, 1536, 97),
    (257, 2560, 128), (1024, 14336, 50),
]
# past 128 rows (two and three row chunks): Q6_K rows the single-pass GEMM does not take
CHUNKED = [(300, 2816, 129), (257, 5632, 192), (130, 4352, 193), (1000, 11008, 256)]


def stream():
    return torch.cuda.current_stream().cuda_stream


def forward(t, qt, x, n, k, rows, ws_bytes=None):
    L = lib()
    out = torch.full((rows, n), float("nan"), dtype=torch.float32, device="cuda")
    need = ctypes.c_size_t(0)
    assert L.qmm_forward(t, None, None, k, None, n, None, 0, ctypes.byref(need), k, n, rows, 0, 0) == 0
    ws = torch.empty(ws_bytes or need.value, dtype=torch.uint8, device="cuda")
    assert L.qmm_forward(t, qt.data_.data_ptr(), x.data_ptr(), k, out.data_ptr(), n, ws.data_ptr(), ws.numel(),
                         ctypes.byref(need), k, n, rows, 1, stream()) == 0
    return out, need.value


@pytest.mark.parametrize("t,n,k,rows", [(t, *s) for t in (qref.Q4_K, qref.Q6_K) for s in SHAPES]
                         + [(qref.Q6_K, *s) for s in CHUNKED]
                         + [(qref.Q4_K, 9000, 1792, 100), (qref.Q6_K, 9000, 4096, 90)])
def test_against_the_oracle_with_slots_and_without(t, n, k, rows):
    rng = np.random.default_rng(zlib.crc32(f"mid-{t}-{n}-{k}-{rows}".encode()))
    wq = qref.from_float(t, weights(rng, n, k))
    qt = QTensor.from_data(wq.tobytes(), (n, k), GgmlDType(t))
    x = rng.standard_normal((rows, k)).astype(np.float32)
    xt = torch.from_numpy(x).cuda()
    print(f"t={t} n={n} k={k} rows={rows}", flush=True)
    y, need = forward(t, qt, xt, n, k, rows)
    assert KERNEL[t] in lib().qmm_last_kernel().decode()
    want = qref.matmul(t, x, wq, n)
    wdeq = qref.to_float(t, wq, n * k).reshape(n, k)
    err = normalised_error(y.cpu().numpy(), want, wdeq, x)
    assert err <= BOUND, err
    # no room for the split slots: the kernels that need none, as exactly
    act = lib().qmm_act_bytes(_lib.ACT_Q8K, k, rows)
    other = no_slots_kernel(t, n, rows) if need > act else KERNEL[t]
    small = forward(t, qt, xt, n, k, rows, act)[0]
    assert other in lib().qmm_last_kernel().decode()
    assert normalised_error(small.cpu().numpy(), want, wdeq, x) <= BOUND
    assert torch.equal(small, y) or need > act
    if need > act:
        assert torch.equal(forward(t, qt, xt, n, k, rows, need - 1)[0], small)
    xq = quantize_act(xt, _lib.ACT_Q8K)
    out = torch.empty_like(y)
    assert lib().qmm_matmul(t, qt.data_.data_ptr(), xq.data_ptr(), out.data_ptr(), n, k, n, rows, stream()) == 0
    assert other in lib().qmm_last_kernel().decode()
    assert torch.equal(out, small)


LARGE = [  # up to 32 rows: the sizes the few-row kernels leave (n, k, rows, taken: of Q4_K, of Q6_K)
    (16390, 512, 17, True, True), (12289, 1280, 32, False, False), (12289, 1536, 17, True, True),
    (12288, 3072, 23, False, True), (8200, 3072, 24, True, True), (8200, 2816, 24, False, True),
    (8200, 7168, 23, False, False), (8192, 4096, 32, False, False), (4100, 7168, 24, True, True),
    (4100, 6912, 32, False, False), (4096, 7168, 32, False, False), (1024, 7168, 24, True, True),
    (1025, 7168, 24, False, False), (1000, 10752, 17, True, True), (1000, 10496, 23, False, False),
    (4096, 13824, 24, True, True), (4096, 13824, 23, False, False), (14336, 4096, 17, True, True),
    (8192, 14336, 17, True, True),
]


@pytest.mark.parametrize("t", [qref.Q4_K, qref.Q6_K], ids=["q4k", "q6k"])
@pytest.mark.parametrize("n,k,rows,q4k,q6k", LARGE)
def test_large_weights_up_to_32_rows(t, n, k, rows, q4k, q6k):
    taken = q4k if t == qref.Q4_K else q6k
    qt = QTensor.quantize(fill_normal(n * k, seed=n + k, std=0.02).reshape(n, k), GgmlDType(t))
    xt = fill_normal(rows * k, seed=rows).reshape(rows, k)
    print(f"t={t} n={n} k={k} rows={rows}", flush=True)
    y, need = forward(t, qt, xt, n, k, rows)
    kernel = lib().qmm_last_kernel().decode()
    few = "launch_sk" if t == qref.Q4_K else "ONE = true" if k >= 2048 else "ONE = false"
    assert (KERNEL[t] if taken else few) in kernel
    x, wdeq = xt.cpu().numpy(), qt.dequantize().cpu().numpy()
    want = qref.matmul(t, x, qt.data_.cpu().numpy(), n)
    err = normalised_error(y.cpu().numpy(), want, wdeq, x)
    assert err <= (BOUND if taken or t == qref.Q4_K else 1e-3), err  # few-row Q6_K: its single-product form
    act = lib().qmm_act_bytes(_lib.ACT_Q8K, k, rows)
    small = forward(t, qt, xt, n, k, rows, act)[0]
    assert torch.equal(small, y) or need > act
    if need > act:
        kernel = lib().qmm_last_kernel().decode()
        assert no_slots_kernel(t, n, rows) in kernel and "ONE = true" not in kernel
        assert normalised_error(small.cpu().numpy(), want, wdeq, x) <= BOUND


LINES = [  # past 32 rows: the Q6_K products the tiled GEMM keeps (n, k, rows, taken here)
    (4096, 1536, 96, True), (8192, 1536, 64, True), (8192, 1536, 65, False), (4100, 2560, 96, True),
    (8200, 2304, 64, False), (8200, 2560, 33, True), (16384, 3840, 65, False), (16384, 4096, 96, True),
    (16390, 1536, 96, True), (4096, 1536, 128, True), (8192, 8192, 97, True), (8200, 8192, 97, False),
    (16390, 8192, 128, True), (32780, 8192, 97, False), (4096, 2304, 129, False),
    (2048, 2304, 129, True), (4096, 2560, 192, True), (4100, 8448, 192, True), (4096, 4352, 193, True),
    (4100, 8448, 193, False),
]


@pytest.mark.parametrize("n,k,rows,taken", LINES)
def test_q6k_lines_to_the_tiled_gemm(n, k, rows, taken):
    """Each side of every line, against the oracle at the first, last and 64
    weight rows between."""
    qt = QTensor.quantize(fill_normal(n * k, seed=n + k, std=0.02).reshape(n, k), GgmlDType.Q6K)
    xt = fill_normal(rows * k, seed=rows).reshape(rows, k)
    print(f"n={n} k={k} rows={rows}", flush=True)
    y = QMatMul(qt).forward(xt)
    assert (KERNEL[qref.Q6_K] if taken else "launch_gemm_q6k(") in lib().qmm_last_kernel().decode()
    some = np.unique(np.linspace(0, n - 1, 66).astype(np.int64))
    wq = np.ascontiguousarray(qt.data_.reshape(-1)[: n * k // 256 * 210].cpu().numpy().reshape(n, -1)[some]).reshape(-1)
    x = xt.cpu().numpy()
    want = qref.matmul(qref.Q6_K, x, wq, len(some))
    wdeq = qref.to_float(qref.Q6_K, wq, len(some) * k).reshape(len(some), k)
    assert normalised_error(y[:, torch.from_numpy(some).cuda()].cpu().numpy(), want, wdeq, x) <= BOUND


@pytest.mark.parametrize("rows", [33, 77, 128])
def test_shared_products_keep_each_weights_bits(rows):
    """Five weights (two launches) of which some are cut and some are not."""
    k = 4096
    mats = []
    for i, n in enumerate((2048, 256, 33, 12000, 130)):
        rng = np.random.default_rng(400 + i)
        wq = qref.from_float(qref.Q4_K, weights(rng, n, k))
        mats.append(QMatMul(QTensor.from_data(wq.tobytes(), (n, k), GgmlDType.Q4K)))
    x = torch.from_numpy(np.random.default_rng(9).standard_normal((rows, k)).astype(np.float32)).cuda()
    for m, y in zip(mats, QMatMul.forward_shared(x, mats)):
        assert torch.equal(y, m.forward(x))


@pytest.mark.parametrize("t,k,ns,rows,launches", [
    (qref.Q4_K, 8192, (8192, 2048, 2048), 24, 2), (qref.Q4_K, 8192, (2048, 8192, 2048), 32, 2),
    (qref.Q6_K, 8192, (8192, 2048, 2048), 32, 2), (qref.Q6_K, 5120, (1024, 5120, 1024), 100, 2),
])
def test_sets_of_which_only_some_weights_are_taken(t, k, ns, rows, launches):
    """Each kernel's weights share its launch (the short-batch kernel's with
    their slots) and keep their own forward's bits."""
    mats = [QMatMul(QTensor.quantize(fill_normal(n * k, seed=40 + i, std=0.02).reshape(n, k), GgmlDType(t)))
            for i, n in enumerate(ns)]
    x = fill_normal(rows * k, seed=rows).reshape(rows, k)
    print(f"t={t} {ns} x {k} rows={rows}", flush=True)
    before = lib().qmm_gemm_launches()
    ys = QMatMul.forward_shared(x, mats)
    assert lib().qmm_gemm_launches() == before + launches
    kernels = set()
    for m, y in zip(mats, ys):
        assert torch.equal(y, m.forward(x))
        kernels.add(KERNEL[t] in lib().qmm_last_kernel().decode())
    assert kernels == {True, False}


@pytest.mark.parametrize("rows", [40, 128])
def test_padded_output_rows_stay_untouched(rows):
    """ldd > n and an n that is no multiple of 4: nothing past a row's n."""
    t, n, k, ldd = qref.Q4_K, 1023, 4096, 1030
    rng = np.random.default_rng(17)
    wq = qref.from_float(t, weights(rng, n, k))
    qt = QTensor.from_data(wq.tobytes(), (n, k), GgmlDType(t))
    x = torch.from_numpy(rng.standard_normal((rows, k)).astype(np.float32)).cuda()
    y, need = forward(t, qt, x, n, k, rows)
    out = torch.full((rows, ldd), float("nan"), dtype=torch.float32, device="cuda")
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    nd = ctypes.c_size_t(0)
    assert lib().qmm_forward(t, qt.data_.data_ptr(), x.data_ptr(), k, out.data_ptr(), ldd, ws.data_ptr(), ws.numel(),
                             ctypes.byref(nd), k, n, rows, 1, stream()) == 0
    assert torch.equal(out[:, :n], y) and bool(torch.isnan(out[:, n:]).all())


def test_q4k_largest_codes_scales_and_mins():
    """Blocks of q = 15 with scales and mins of 63 (sc q = 945, the largest
    operand products 105) against rows of one sign (|T| near 2^24.9, |Tm| near
    2^21), the quantizer's edge rows, and rows scaled by 1e-30 and 1e30."""
    n, k = 64, 2048
    rng = np.random.default_rng(77)
    wq = qref.from_float(qref.Q4_K, weights(rng, n, k)).view(np.uint8).reshape(n * k // 256, 144).copy()
    # get_scale_min_k4's packing of 63 everywhere is all ones
    wq[::2, 4:16] = 0xFF
    wq[::2, 16:] = 0xFF
    wq = wq.reshape(-1)
    qt = QTensor.from_data(wq.tobytes(), (n, k), GgmlDType.Q4K)
    sp = special_rows(k)
    x = np.concatenate([sp, np.full((3, k), 1.0, np.float32), rng.standard_normal((30, k)).astype(np.float32)])
    x[len(sp) + 1] *= -1.0
    x[-1] *= np.float32(1e-30)
    x[-2] *= np.float32(1e30)
    y = QMatMul(qt).forward(torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.all(y[0] == 0.0)
    want = qref.matmul(qref.Q4_K, x, wq, n)
    wdeq = qref.to_float(qref.Q4_K, wq, n * k).reshape(n, k)
    assert normalised_error(y, want, wdeq, x) <= BOUND
