"""Winograd convolutions whose reduction is cut into ranges of the input channels (few work items, many channels) against
the uncut launch and fp64: squares, stacked batches and their pieces, a last block of output channels that is not full,
pooling, output masks, ranges that take the fp32 products.

Bound: the ranges' errors are the uncut kernel's at most (4.5e-7 of the result in the 2-norm at 512 channels, less for
shorter sums), and the sum of up to eight ranges adds seven roundings of 2^-24 (a 2-norm of 1.6e-7 if each were half an
ulp of the whole)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CL = torch.channels_last
SHAPES = [(1, 256, 64, 14, 14), (2, 512, 512, 14, 14), (8, 512, 512, 14, 14), (3, 256, 100, 9, 23), (2, 384, 192, 28, 28),
          (2, 256, 256, 20, 56), (1, 512, 68, 30, 16), (4, 1024, 64, 7, 7), (5, 256, 64, 12, 8), (3, 512, 128, 18, 12)]


def _operands(N, C, K, H, W, seed=0):
    g = torch.Generator().manual_seed(seed + N + C + K)
    x = torch.randn(N, C, H, W, generator=g).cuda().contiguous(memory_format=CL)
    w = (torch.randn(K, C, 3, 3, generator=g) * (2.0 / (9 * C)) ** 0.5).cuda().contiguous(memory_format=CL)
    return x, w, torch.randn(K, generator=g).cuda()


def _exact(x, w):
    return torch.nn.functional.conv2d(x.cpu().double(), w.cpu().double(), padding=1)


def _uncut(monkeypatch, call):
    from pipedream_amd import ops
    with monkeypatch.context() as m:
        m.setattr(ops, "_conv_split_bytes", lambda *args: 0)
        return call()


def _rel(a, b):
    return float((a.cpu().double() - b.cpu().double()).norm() / b.cpu().double().norm())


@pytest.mark.parametrize("N,C,K,H,W", SHAPES)
def test_forward_pool_and_input_gradient(monkeypatch, N, C, K, H, W):
    from pipedream_amd import ops
    assert ops._conv_split_bytes(N, H, W, C, K) > 0
    x, w, bias = _operands(N, C, K, H, W)
    want = _exact(x, w)
    y = ops.conv3x3_forward(x, w)
    whole = _uncut(monkeypatch, lambda: ops.conv3x3_forward(x, w))
    assert _rel(y, want) <= max(1.1 * _rel(whole, want), 2e-7)
    assert torch.equal(y, ops.conv3x3_forward(x, w))
    biased = ops.conv3x3_forward(x, w, bias, relu=True)
    assert torch.equal(biased, torch.relu(y + bias[:, None, None]))
    if H >= 2 and W >= 2:
        pooled, idx = ops.conv3x3_forward_pool(x, w, bias, relu=True)
        p2, i2 = ops.maxpool2x2_idx(biased)
        assert torch.equal(pooled, p2) and torch.equal(idx, i2)
    # input gradient (K channels are reduced over), with the ReLU mask of the layer in front
    if K % 16 == 0 and ops._conv_split_bytes(N, H, W, K, C) > 0:
        dy = torch.randn(N, K, H, W).cuda().contiguous(memory_format=CL)
        act = torch.randn(N, C, H, W).cuda().contiguous(memory_format=CL)
        dx = ops.conv3x3_input_grad(dy, w, x_rectified=act)
        ref = torch.nn.grad.conv2d_input((N, C, H, W), w.cpu().double(), dy.cpu().double(), padding=1) * (act.cpu() > 0)
        whole = _uncut(monkeypatch, lambda: ops.conv3x3_input_grad(dy, w, x_rectified=act))
        assert _rel(dx, ref) <= max(1.1 * _rel(whole, ref), 2e-7)


def test_ranges_that_f16_does_not_hold(monkeypatch):
    """Infinities, zero kernels and outlying pixels in some ranges only."""
    from pipedream_amd import ops
    x, w, _ = _operands(2, 512, 128, 14, 14)
    w[70, 300] = 0
    x[1, 200:260, 3, 3] *= 2.0 ** 20
    want = _exact(x, w)
    assert _rel(ops.conv3x3_forward(x, w), want) < 1e-6
    x[0, 17, 6, 6] = float("inf")
    y = ops.conv3x3_forward(x, w)
    whole = _uncut(monkeypatch, lambda: ops.conv3x3_forward(x, w))
    assert torch.equal(torch.isfinite(y), torch.isfinite(whole)) and torch.equal(torch.isnan(y), torch.isnan(whole))
    ok = torch.isfinite(whole)
    torch.testing.assert_close(y[ok], whole[ok], rtol=1e-4, atol=float(whole[ok].abs().max()) * 1e-6)


def test_many_items_are_not_cut():
    from pipedream_amd import ops
    assert ops._conv_split_bytes(64, 14, 14, 512, 512) == 0 and ops._conv_split_bytes(1, 14, 14, 64, 512) == 0
