"""The multi-row decode kernel of the 32-value formats at the lines between one
and two weight rows a wave (4096 weight rows from 7 activation rows, 8192 from
4): every activation row has the bits of its own 1-row product."""
import pytest
import torch

from swarmllm_amd import GgmlDType, QMatMul, QTensor, fill_normal

pytestmark = pytest.mark.gpu


def weight(name, n, k, seed):
    blocks = n * k // 32
    g = torch.Generator("cuda").manual_seed(seed)
    size = {"Q8_0": 34, "Iq4Nl": 18, "Mxfp4": 17}[name]
    b = torch.randint(0, 256, (blocks, size), dtype=torch.uint8, device="cuda", generator=g)
    if name == "Mxfp4":
        b[:, 0] = 118 + b[:, 0] % 8
    else:
        b[:, :2] = torch.rand(blocks, 1, device="cuda", generator=g).add(0.5).mul(0.01).half().view(torch.uint8)
    return QTensor(b.reshape(-1), (n, k), getattr(GgmlDType, name))


@pytest.mark.parametrize("name", ["Q8_0", "Iq4Nl", "Mxfp4"])
@pytest.mark.parametrize("rows,n", [(8, 4095), (7, 4097), (6, 4097), (4, 8191), (5, 8193), (3, 8193)])
def test_rows_have_their_own_bits(name, rows, n):
    k = 352  # a partial span of 11 blocks
    q = QMatMul(weight(name, n, k, n + rows))
    x = fill_normal(rows * k, seed=rows).reshape(rows, k)
    y = q.forward(x)
    for r in range(rows):
        assert torch.equal(y[r], q.forward(x[r:r + 1])[0]), f"row {r}"
