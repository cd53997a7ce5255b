"""The LSTM time loop whose recurrent products run on the bf16 matrix pipes (pd_lstm_f32x6.hip) against a 64-bit
evaluation of the same layer, at the edges of its tiles: 16 rows of a row tile, 64 of a row block, eight waves that
share the chunks of 32 k (fewer chunks than waves, chunks that do not divide).

Bound: a gate sum of H products and three other terms of size O(1) carries at most (H / 16 + 16) roundings of 2^-24 of
the running sum; the recurrence of T steps adds them up with gain at most one (the weights' rows sum to less than
one in size), so 2-norm errors stay below T (H / 16 + 16) 2^-24 / 4 -- the roundings being independent, far below."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(T, B, H, seed=3):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, B, 8, generator=g)
    w_ih, w_hh = torch.randn(4 * H, 8, generator=g) * 0.2, (torch.rand(4 * H, H, generator=g) * 2 - 1) / H ** 0.5
    b_ih, b_hh = torch.randn(4 * H, generator=g) * 0.1, torch.randn(4 * H, generator=g) * 0.1
    return [t.cuda() for t in (x, w_ih, w_hh, b_ih, b_hh)], torch.randn(T, B, H, generator=g).cuda()


def _in_64_bits(params, dy):
    x, w_ih, w_hh, b_ih, b_hh = (t.double().requires_grad_() for t in params)
    H = w_hh.shape[1]
    h = c = torch.zeros(x.shape[1], H, dtype=torch.double, device=x.device)
    ys = []
    for t in range(x.shape[0]):
        i, f, g, o = (x[t] @ w_ih.t() + h @ w_hh.t() + b_ih + b_hh).split(H, 1)
        c = f.sigmoid() * c + i.sigmoid() * g.tanh()
        h = o.sigmoid() * c.tanh()
        ys.append(h)
    y = torch.stack(ys)
    y.backward(dy.double())
    return y.detach(), x.grad, w_ih.grad, w_hh.grad, b_ih.grad


@pytest.mark.parametrize("B,H", [(1, 32), (16, 64), (17, 96), (33, 32), (48, 160), (49, 288), (64, 64), (65, 32), (100, 544),
                                 (128, 256), (40, 1024), (128, 1024)])
def test_layer_matches_64_bits(B, H):
    from pipedream_amd import ops, _cabi
    assert _cabi.lib().pd_lstm_f32x6_supported(B, H)
    T = 4
    params, dy = _layer(T, B, H)
    y, (gates, c) = ops.lstm_forward(*params)
    x, w_ih, w_hh = params[:3]
    got = (y,) + tuple(ops.lstm_backward(dy, x, y, gates, c, w_ih, w_hh))
    bound = T * (H / 16 + 16) * 2.0 ** -24 / 4
    for a, b in zip(got, _in_64_bits(params, dy)):
        assert float((a.double() - b).norm() / b.norm()) < bound


def test_shapes_outside_the_tiles_take_the_other_loop():
    from pipedream_amd import _cabi
    lib = _cabi.lib()
    assert not any(lib.pd_lstm_f32x6_supported(B, H) for B, H in ((129, 64), (8, 48), (0, 64), (8, 8224)))


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38])
def test_weights_that_have_no_terms(value):
    """An infinity, a NaN or a value that rounds to infinity in bf16: what the fp32 MFMA loop gives, NaNs included."""
    from pipedream_amd import ops
    params, dy = _layer(3, 20, 64)
    params[2][5, 7] = value
    x, w_ih, w_hh = params[:3]

    def run():
        y, (gates, c) = ops.lstm_forward(*params)
        return (y, gates, c) + tuple(ops.lstm_backward(dy, x, y, gates, c, w_ih, w_hh))
    got = run()
    ops.set_gemm_f32_algorithm("mfma_f32")
    try:
        want = run()
    finally:
        ops.set_gemm_f32_algorithm("auto")
    for a, b in zip(got[:3], want[:3]):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-6, equal_nan=True)
    for a, b in zip(got[3:], want[3:]):
        assert torch.equal(torch.isfinite(a), torch.isfinite(b))
