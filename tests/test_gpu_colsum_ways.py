"""The second launch of a batch of column sums at the number of rows where its blocks get four times as many waves: the same
bits either way (a longer matrix in the batch decides for all of them), and 64-bit sums.

Bound: at most 32 + 5 additions per chain and tree for the lengths here, each rounded to 2^-24 of a partial sum."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _sums(mats):
    from pipedream_amd import ops
    batch = ops.ColsumBatch()
    outs = [torch.full((m.size(1),), float("nan"), device="cuda") for m in mats]
    for m, o in zip(mats, outs):
        batch.add(m, o, 0.0)
    batch.run()
    return outs


@pytest.mark.parametrize("rows", [1, 3, 31, 32, 33, 64, 127, 128, 129, 255])
@pytest.mark.parametrize("cols", [1, 63, 65, 200])
def test_either_number_of_waves_gives_the_same_bits(rows, cols):
    g = torch.Generator().manual_seed(rows * 1000 + cols)
    x = torch.randn(rows, cols, generator=g).cuda()
    y = torch.randn(rows, cols, generator=g).bfloat16().cuda()       # 64 ranges of rows in the first launch
    alone, beside = _sums([x, y]), _sums([x, y, torch.ones(129, 8, device="cuda")])
    assert torch.equal(alone[0], beside[0]) and torch.equal(alone[1], beside[1])
    assert torch.equal(beside[2], torch.full((8,), 129.0, device="cuda"))
    for got, m in zip(alone, (x, y)):
        bound = 37 * 2.0 ** -24 * m.double().abs().sum(0)
        assert bool(((got.double() - m.double().sum(0)).abs() <= bound).all())
