"""bf16 products at the edges of the kernels' tiles (32 to 256 rows and columns), of their rings (chunks of 32 k, rounds of
128) and of the epilogue's row blocks, in all four layouts, against fp64 of the same bf16 operands.

Bound: products of bf16 values are exact in fp32, a running sum is rounded once per 16 k and eight sums are added up at
most: |error| <= (K / 16 + 16) 2^-24 sum |a| |b|, and for a bf16 result 2^-8 of its value."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def _operand(rows, cols, g, pad=8):
    """A matrix with NaNs behind every row and below the last one: nothing outside may be read as a value."""
    big = torch.full((rows + 40, cols + pad), float("nan"), dtype=BF)
    big[:rows, :cols] = torch.randn(rows, cols, generator=g).to(BF)
    return big.cuda()[:rows, :cols]


def _case(M, N, K, ta, tb, seed=0):
    g = torch.Generator().manual_seed(seed + M + N + K)
    a, b = _operand(*((K, M) if ta else (M, K)), g), _operand(*((N, K) if tb else (K, N)), g)
    ad, bd = (a.t() if ta else a).double(), (b.t() if tb else b).double()
    return a, b, ad @ bd, (K / 16 + 16) * 2.0 ** -24 * (ad.abs() @ bd.abs())


SHAPES = [(8, 8, 8), (32, 64, 40), (64, 64, 128), (72, 56, 136), (64, 72, 3000), (88, 768, 768), (128, 128, 120), (136, 264, 600),
          (200, 2304, 88), (600, 776, 200), (600, 3072, 256), (256, 1032, 1032), (1240, 1024, 72), (1920, 512, 512), (4096, 4104, 128),
          (4040, 4096, 256), (64, 192, 4096), (640, 264, 2080), (200, 328, 7200),
          # reductions of at most 192: staged, in tiles of 128 x 128 from 256 of them on
          (72, 56, 8), (136, 2056, 64), (2056, 2056, 40), (2040, 2056, 192), (4104, 1032, 136), (2056, 2056, 200),
          # staged 256 x 256 from 192 tiles on, whatever 128 leaves of k; staged 128 x 128 of longer reductions
          (4104, 3080, 40), (4104, 3080, 136), (4096, 3072, 328), (2312, 2056, 712),
          # ragged reductions of few tiles and, for B as [K][N], long ones of more, over the waves of a block
          (304, 520, 160), (104, 1000, 800), (304, 1024, 1056)]


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product(M, N, K, ta, tb):
    from pipedream_amd import ops
    a, b, ref, bound = _case(M, N, K, ta, tb)
    start = torch.randn(M, N).cuda()
    out = start.clone()
    ops.gemm_bf16(a, b, trans_a=bool(ta), trans_b=bool(tb), out=out, beta=1.0)
    assert bool(((out.double() - ref - start.double()).abs() <= bound + 2.0 ** -22 * (ref.abs() + start.double().abs())).all())
    y = ops.gemm_bf16(a, b, trans_a=bool(ta), trans_b=bool(tb))
    assert bool(((y.double() - ref).abs() <= bound + 2.0 ** -8 * ref.abs()).all())


@pytest.mark.parametrize("M,N,K", [(72, 56, 136), (88, 768, 768), (600, 776, 200), (600, 3072, 256), (1240, 1024, 72), (640, 264, 2080),
                                   (4040, 4096, 256)])
def test_epilogues(M, N, K):
    """Bias, residual, GELU and its derivative in tiles that stick out of the matrix; what lies behind the rows stays."""
    from pipedream_amd import ops
    a, b, ref, bound = _case(M, N, K, 0, 1)
    bias, res = torch.randn(N).cuda(), torch.randn(M, N).to(BF).cuda()
    wide = torch.zeros(M + 8, N + 8, dtype=BF).cuda()
    ops.gemm_bf16(a, b, trans_b=True, bias=bias, residual=res, out=wide[:M, :N])
    want = ref + bias.double() + res.double()
    slack = bound + 2.0 ** -22 * (ref.abs() + bias.double().abs())
    assert bool(((wide[:M, :N].double() - want).abs() <= slack + 2.0 ** -8 * want.abs()).all())
    assert not wide[M:].any() and not wide[:, N:].any()
    f, g = ops.gemm_bf16_gelu(a, b, trans_b=True, bias=bias)
    assert bool(((f.double() - ref - bias.double()).abs() <= slack + 2.0 ** -8 * (ref + bias.double()).abs()).all())
    torch.testing.assert_close(g.float(), torch.nn.functional.gelu(f.float()), rtol=2.0 ** -7, atol=2e-6)
    w = b.t().contiguous()
    df = ops.gemm_bf16_gelu_backward(a, w, f)
    fr = f.double().requires_grad_()
    torch.nn.functional.gelu(fr).sum().backward()
    want = ref * fr.grad
    assert bool(((df.double() - want).abs() <= (bound + 2.0 ** -8 * ref.abs()) * (fr.grad.abs() + 1e-6) + 2.0 ** -8 * want.abs() + 1e-6 * ref.abs()).all())


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("batch,M,N,K", [(300, 64, 64, 128), (520, 40, 32, 40), (130, 136, 64, 264), (80, 200, 24, 200),
                                         (260, 72, 128, 64), (130, 136, 136, 192), (257, 64, 72, 128), (80, 1032, 48, 256),
                                         (200, 200, 200, 96)])
def test_batches_of_small_products(batch, M, N, K, ta, tb):
    """Attention's products at head dimensions without a fused kernel: many entries, narrow sides, short reductions."""
    from pipedream_amd import ops
    g = torch.Generator().manual_seed(batch + M)
    a = torch.randn(*((batch, K, M) if ta else (batch, M, K)), generator=g).to(BF).cuda()
    b = torch.randn(*((batch, N, K) if tb else (batch, K, N)), generator=g).to(BF).cuda()
    out = torch.full((batch * M + 8, N), float("nan"), dtype=BF, device="cuda")
    ops._batched(ta, tb, M, N, K, a, 0, a.size(2), b, 0, b.size(2), out, 0, N, 1.0, batch, 1, (M * K, 0, N * K, 0, M * N, 0))
    ad, bd = (a.transpose(1, 2) if ta else a).double().contiguous(), (b.transpose(1, 2) if tb else b).double().contiguous()
    ref = torch.bmm(ad, bd)
    bound = (K / 16 + 16) * 2.0 ** -24 * torch.bmm(ad.abs(), bd.abs()) + 2.0 ** -8 * ref.abs()
    assert bool(((out[:batch * M].view(batch, M, N).double() - ref).abs() <= bound).all())
    assert torch.isnan(out[batch * M:].float()).all()


@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("far", ["a", "b"])
def test_rows_far_apart(far, ta, tb):
    """Leading dimensions of 2^22 elements: the kernel that stages through registers, whose offsets are 64 bits wide, for a
    reduction that the direct-to-LDS kernels would otherwise have taken."""
    from pipedream_amd import ops
    g = torch.Generator().manual_seed(3)
    M, N, K = 24, 72, 328

    def operand(rows, cols, wide):
        t = torch.randn(rows, cols, generator=g).to(BF).cuda()
        if not wide:
            return t
        big = torch.full((rows, 1 << 22), float("nan"), dtype=BF, device="cuda")
        big[:, :cols] = t
        return big[:, :cols]
    a = operand(*((K, M) if ta else (M, K)), far == "a")
    b = operand(*((N, K) if tb else (K, N)), far == "b")
    y = ops.gemm_bf16(a, b, trans_a=bool(ta), trans_b=bool(tb), out_f32=True)
    ad, bd = (a.t() if ta else a).double(), (b.t() if tb else b).double()
    bound = (K / 16 + 16) * 2.0 ** -24 * (ad.abs() @ bd.abs())
    assert bool(((y.double() - ad @ bd).abs() <= bound).all())
