"""The Q8_0 / IQ4_NL / MXFP4 GEMM (gemm_b32.hip) at the edges of its
workgroup shapes (32, 64 and 128 rows; 32 and 64 weight rows; one to eight K
ranges), of its 4-block stages (whole stages with 16-byte aligned rows take
offsets only a scalar moves, the others clamped ones) and with activation
scales that overflow f16.

Bound: every block sum is an exact integer and every scale product of two f16
numbers exact in f32, so a result, like the oracle's, is off by one rounding a
block and one per addition: each at most (nb + 8) 2^-24 of the sum of the
terms' magnitudes, which is at most ||w|| ||x|| (of the quantized x, within 1%).
Their difference is within 1e-5 up to 75 blocks and 1.7e-5 at 128; 1e-5 is held
(1e-7 measured)."""
import zlib

import numpy as np
import pytest
import torch

from helpers import TYPES, normalised_error, weights
from oracle import qref
from swarmllm_amd import GgmlDType, QMatMul, QTensor
from swarmllm_amd._lib import lib

pytestmark = pytest.mark.gpu

FORMATS = ["Q8_0", "IQ4_NL", "MXFP4"]
SHAPES = [  # (n, k, rows)
    (31, 32, 9), (33, 64, 32), (65, 160, 33), (64, 128, 64), (8200, 96, 40), (63, 1024, 65), (200, 2880, 128),
    (12300, 128, 129), (33000, 64, 100), (1000, 4096, 200), (512, 992, 300),
]


def make(name, n, k, seed):
    w = weights(np.random.default_rng(seed), n, k)
    wq = qref.from_float(TYPES[name], w)
    return QMatMul(QTensor.from_data(wq.tobytes(), (n, k), GgmlDType(TYPES[name]))), wq


@pytest.mark.parametrize("name", FORMATS)
@pytest.mark.parametrize("n,k,rows", SHAPES)
def test_against_the_oracle(name, n, k, rows):
    seed = zlib.crc32(f"b32-{name}-{n}-{k}-{rows}".encode())
    mm, wq = make(name, n, k, seed)
    x = np.random.default_rng(seed + 1).standard_normal((rows, k)).astype(np.float32)
    print(f"{name} n={n} k={k} rows={rows}", flush=True)
    y = mm.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    assert "launch_gemm_b32(" in lib().qmm_last_kernel().decode()
    want = qref.matmul(TYPES[name], x, wq, n)
    wdeq = qref.to_float(TYPES[name], wq, n * k).reshape(n, k)
    assert normalised_error(y, want, wdeq, x) <= 1e-5


# the 128-row shapes past their first stages: uncut (512 tiles and more) and in
# two K ranges (192 and more); whole stages and a partial last one, an odd
# number of stages, of which the second range has one
@pytest.mark.parametrize("name", FORMATS)
@pytest.mark.parametrize("n,k,rows", [(33000, 1024, 100), (33000, 416, 100), (12300, 1024, 129), (12300, 416, 129),
                                      (12300, 352, 200)])
def test_128_row_shapes_over_many_stages(name, n, k, rows):
    """Against the oracle at the first, last and 130 weight rows between; two
    rows have f16 block scales below the normal range and near its top."""
    seed = zlib.crc32(f"b32-{name}-{n}-{k}-{rows}".encode())
    mm, wq = make(name, n, k, seed)
    x = np.random.default_rng(seed + 1).standard_normal((rows, k)).astype(np.float32)
    x[5] *= np.float32(1e-4)
    x[6] *= np.float32(1e6)
    print(f"{name} n={n} k={k} rows={rows}", flush=True)
    y = mm.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    assert "launch_gemm_b32(" in lib().qmm_last_kernel().decode()
    some = np.unique(np.linspace(0, n - 1, 132).astype(np.int64))
    part = np.ascontiguousarray(wq.view(np.uint8).reshape(n, -1)[some]).reshape(-1)
    want = qref.matmul(TYPES[name], x, part, len(some))
    wdeq = qref.to_float(TYPES[name], part, len(some) * k).reshape(len(some), k)
    assert normalised_error(y[:, some], want, wdeq, x) <= 1e-5


@pytest.mark.parametrize("name", FORMATS)
@pytest.mark.parametrize("rows", [20, 64, 140])
def test_shared_products_of_several_shapes_keep_each_weights_bits(name, rows):
    k = 1024
    mats = [make(name, n, k, 30 + i)[0] for i, n in enumerate((40, 9000, 700, 33000, 64))]
    x = torch.from_numpy(np.random.default_rng(5).standard_normal((rows, k)).astype(np.float32)).cuda()
    for m, y in zip(mats, QMatMul.forward_shared(x, mats)):
        assert torch.equal(y, m.forward(x))


@pytest.mark.parametrize("name", FORMATS)
@pytest.mark.parametrize("rows", [12, 70])
def test_an_overflowing_activation_scale_stays_in_its_row(name, rows):
    """A block of 1e9 has the f16 scale inf (in the reference as here): its
    row is infinite or NaN exactly where the decode kernel's is (the oracle's
    AVX2 lanes add infinities of both signs), every other row finite."""
    n, k = 96, 256
    mm, _ = make(name, n, k, 8)
    x = np.random.default_rng(9).standard_normal((rows, k)).astype(np.float32)
    x[3, 64:96] *= np.float32(1e9)
    y = mm.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    one = mm.forward(torch.from_numpy(x[3:4]).cuda()).cpu().numpy()[0]
    others = [r for r in range(rows) if r != 3]
    assert np.isfinite(y[others]).all()
    assert not np.isfinite(y[3]).any()
    assert np.array_equal(np.isnan(y[3]), np.isnan(one)) and np.array_equal(y[3] > 0, one > 0)
