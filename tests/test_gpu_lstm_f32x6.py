"""The LSTM time loop whose recurrent products run on the bf16 matrix pipes (pd_lstm_f32x6.hip) against a 64-bit
evaluation of the same layer, at the edges of its tiles: 16 rows of a row tile, 64 of a row block, eight waves that
share the chunks of 32 k (fewer chunks than waves, chunks that do not divide).

Bound: fp32 accuracy is what the fp32 MFMA loop has on the same operands: no 2-norm error against 64 bits more than 1.2
times its (0.4 to 1.04 times measured).  With any one of the three small products of the split left out the error of y
is 2.3e-7 at least, and 8e-7 where the recurrent product outweighs the other terms (weights times 4); the fp32 loop's are
1e-7 and at most 1.8e-7."""
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


def _run(params, dy):
    from pipedream_amd import ops
    y, (gates, c) = ops.lstm_forward(*params)
    return (y,) + tuple(ops.lstm_backward(dy, params[0], y, gates, c, params[1], params[2]))


def _no_worse_than_fp32(params, dy):
    from pipedream_amd import ops
    got, exact = _run(params, dy), _in_64_bits(params, dy)
    ops.set_gemm_f32_algorithm("mfma_f32")
    try:
        fp32 = _run(params, dy)
    finally:
        ops.set_gemm_f32_algorithm("auto")
    for name, a, b, c in zip(("y", "dx", "dw_ih", "dw_hh", "db"), got, fp32, exact):
        error, allowed = (float((t.double() - c).norm() / c.norm()) for t in (a, b))
        assert error <= 1.2 * allowed, (name, error, allowed)


@pytest.mark.parametrize("scale", [1, 4])
@pytest.mark.parametrize("B,H", [(1, 32), (16, 64), (17, 96), (33, 32), (48, 160), (49, 288), (64, 64), (65, 32), (100, 544),
                                 (128, 256), (40, 1024), (128, 1024)])
def test_layer_matches_64_bits(B, H, scale):
    from pipedream_amd import _cabi
    assert _cabi.lib().pd_lstm_f32x6_supported(B, H)
    params, dy = _layer(5, B, H)
    params[2] *= scale
    _no_worse_than_fp32(params, dy)


@pytest.mark.parametrize("T,B,H", [(50, 128, 256), (31, 40, 512), (40, 16, 96)])
def test_rounding_has_no_direction(T, B, H):
    """The bias gradients add up thousands of results: an error of one sign in each of them would not stay small (2.9 times the
    fp32 loop's over 50 steps of 128 rows where every sum is rounded towards minus infinity)."""
    _no_worse_than_fp32(*_layer(T, B, H))


@pytest.mark.parametrize("T,B,H", [(6, 129, 64), (5, 7, 48), (4, 200, 96)])
def test_shapes_outside_the_tiles_take_the_other_loop(T, B, H):
    """Bound: a gate sum carries at most H / 4 + 16 roundings of 2^-24 of its running sum, T of them follow each other, and
    errors that are independent add up as the root of their number: 4 sqrt(T (H / 4 + 16)) 2^-24."""
    from pipedream_amd import _cabi
    assert not _cabi.lib().pd_lstm_f32x6_supported(B, H)
    params, dy = _layer(T, B, H)
    for a, b in zip(_run(params, dy), _in_64_bits(params, dy)):
        assert float((a.double() - b).norm() / b.norm()) < 4 * (T * (H / 4 + 16)) ** 0.5 * 2.0 ** -24


def test_supported_shapes():
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
