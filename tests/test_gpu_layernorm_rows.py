"""LayerNorm with all of a row's loads in flight: 1, 2 and 4 vectors of 8 per lane (rows of up to 512, 1024, 2048), rows that
end inside a vector's lanes, a last block of fewer than eight rows, with and without the residual gradient.

Bound: fp32 arithmetic, one rounding to bf16 on the way out: 2^-9 in the 2-norm, as the inputs are exact; twice that where a
rounded residual sum cancels.  dgamma / dbeta are fp32 sums of at most 41 rows of products: 1e-5."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float((a.double().cpu() - b.double().cpu()).norm() / b.double().cpu().norm())


@pytest.mark.parametrize("M", [1, 7, 8, 9, 41])
@pytest.mark.parametrize("H", [8, 504, 512, 520, 768, 1024, 1032, 1536, 2048])
def test_layernorm(M, H):
    from pipedream_amd import ops
    g = torch.Generator().manual_seed(M * 4099 + H)
    x, dy, res = ((torch.randn(M, H, generator=g) * 2 + 0.5).bfloat16() for _ in range(3))
    gamma, beta = torch.randn(H, generator=g), torch.randn(H, generator=g)
    xd, gd, bd = x.double().requires_grad_(), gamma.double().requires_grad_(), beta.double().requires_grad_()
    ref = F.layer_norm(xd, (H,), gd, bd, 1e-5)
    ref.backward(dy.double())
    y, mean, rstd = ops.layernorm_forward(x.cuda(), gamma.cuda(), beta.cuda(), 1e-5)
    assert _rel(y, ref.detach()) < 2.0 ** -8
    dx, dg, db = ops.layernorm_backward(dy.cuda(), x.cuda(), gamma.cuda(), mean, rstd)
    assert _rel(dx, xd.grad) < 2.0 ** -8 and _rel(dg, gd.grad) < 1e-5 and _rel(db, bd.grad) < 1e-5
    dxr, dg2, db2 = ops.layernorm_backward(dy.cuda(), x.cuda(), gamma.cuda(), mean, rstd, residual=res.cuda())
    assert _rel(dxr, xd.grad + res.double()) < 2.0 ** -8
    assert torch.equal(dg, dg2) and torch.equal(db, db2)
