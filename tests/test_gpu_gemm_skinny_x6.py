"""Products of at most 128 rows on the bf16 matrix pipes (pd_gemm_skinny_f32x6.hip) against 64 bits, at the edges of its
tiles: 16 rows, blocks of 64, blocks of 32 and 64 columns, chunks of 32 k over eight waves and a last one that is partly
empty, one range of k and several.

Bound: each operand is the exact sum of its terms, the products left out are below 2^-24 of a product, and a wave's sum
is rounded once per MFMA (six per 32 k), the sums over waves and ranges fewer than 64 times: |error| <=
(6 K / 32 / 8 + 64 + 2) 2^-24 sum |a| |b| whatever the split.  That the small products are there shows in the 2-norm: no
more than the fp32 MFMA kernels' error on the same operands (0.3 to 0.86 of it measured, at most 6e-7; without one of the
products 1.1e-6 at least)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 8), (16, 4, 32), (17, 36, 40), (31, 100, 256), (32, 64, 264), (48, 1028, 72), (49, 32, 2048), (64, 516, 1096),
          (65, 1000, 128), (128, 132, 3080), (100, 2052, 520), (8, 4096, 4104), (40, 260, 1000), (24, 516, 904)]


@pytest.fixture(autouse=True)
def _any_weights(monkeypatch):
    from pipedream_amd import ops
    monkeypatch.setattr(ops, "SKINNY_X6_MIN_WEIGHTS", 0)
    monkeypatch.setattr(ops, "_skinny_x6_min_k", lambda M, trans_b: 0)


def _operands(M, N, K, trans_b, seed=1):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K, generator=g).cuda()
    b = torch.randn(*((N, K) if trans_b else (K, N)), generator=g).cuda()
    return a, b, (b.t() if trans_b else b).double()


def _fp32(a, b, trans_b):
    from pipedream_amd import ops
    ops.set_gemm_f32_algorithm("mfma_f32")
    try:
        return ops.gemm(a, b, trans_b=trans_b)
    finally:
        ops.set_gemm_f32_algorithm("auto")


def _error(got, exact):
    return float((got.double() - exact).norm() / exact.norm())


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,N,K", [(16, 512, 512), (64, 4096, 1096), (128, 2048, 2048), (32, 1024, 64), (33, 2052, 128)])
def test_rounding_has_no_direction(M, N, K, trans_b):
    """Sums over the rows and over the columns of the result, which add up errors of one sign (3 to 7 times the fp32 kernels'
    row sums where every addition is rounded towards minus infinity): 1.2 times the fp32 kernels' errors."""
    from pipedream_amd import ops
    a, b, bd = _operands(M, N, K, trans_b)
    ref, got, fp32 = a.double() @ bd, ops.gemm(a, b, trans_b=trans_b).double(), _fp32(a, b, trans_b).double()
    for dim in (0, 1):
        assert _error(got.sum(dim), ref.sum(dim)) <= 1.2 * _error(fp32.sum(dim), ref.sum(dim)), dim


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_product_matches_64_bits(M, N, K, trans_b):
    from pipedream_amd import ops
    a, b, bd = _operands(M, N, K, trans_b)
    bias = torch.randn(N).cuda()
    start = torch.randn(M, N).cuda()
    out = start.clone()
    assert ops._use_skinny_x6(M, N, K, False, trans_b, a, b, a.stride(0), b.stride(0))
    ops.gemm(a, b, trans_b=trans_b, bias=bias, out=out, beta=0.5)
    ref = a.double() @ bd
    bound = (6 * K / 256 + 66) * 2.0 ** -24 * (a.double().abs() @ bd.abs()) + 2.0 ** -22 * (bias.abs() + start.abs() + ref.abs())
    assert bool(((out.double() - (ref + bias + 0.5 * start)).abs() <= bound).all())
    assert _error(ops.gemm(a, b, trans_b=trans_b), ref) <= _error(_fp32(a, b, trans_b), ref)
    got = ops.gemm(a, b, trans_b=trans_b, relu=True)
    assert bool(((got.double() - ref.clamp(min=0)).abs() <= bound).all()) and bool((got >= 0).all())


def test_rows_apart_odd_widths_and_offset_outputs():
    """Leading dimensions beyond the row, an N that 4 does not divide and an unaligned bias or output: one range of k."""
    from pipedream_amd import ops
    g = torch.Generator().manual_seed(2)
    a = torch.randn(20, 4000, generator=g).cuda()[:, :2048]
    b = torch.randn(70, 2056, generator=g).cuda()[:, :2048]
    ref = a.double() @ b.double().t()
    bound = (6 * 2048 / 256 + 66) * 2.0 ** -24 * (a.double().abs() @ b.double().abs().t())
    wide = torch.zeros(20, 101).cuda()
    ops.gemm(a, b, trans_b=True, out=wide[:, 1:71])
    assert bool(((wide[:, 1:71].double() - ref).abs() <= bound).all()) and not wide[:, 71:].any() and not wide[:, 0].any()
    bias = torch.randn(69, generator=g).cuda()[1:]
    got = ops.gemm(a, b[:68], trans_b=True, bias=bias)
    assert bool(((got.double() - ref[:, :68] - bias).abs() <= bound[:, :68] + 2.0 ** -22 * (ref[:, :68].abs() + bias.abs())).all())


@pytest.mark.parametrize("trans_b", [False, True])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.4e38])
def test_operands_that_have_no_terms(value, trans_b):
    """What the fp32 MFMA kernels give, NaNs included (K = 2056: the last chunk is partly empty, several ranges)."""
    from pipedream_amd import ops
    a, b, _ = _operands(33, 68, 2056, trans_b)
    a[3, 2055] = value
    b[5, 7] = value
    b[(9, 2050) if trans_b else (2050, 9)] = value
    got = ops.gemm(a, b, trans_b=trans_b)
    ops.set_gemm_f32_algorithm("mfma_f32")
    try:
        want = ops.gemm(a, b, trans_b=trans_b)
    finally:
        ops.set_gemm_f32_algorithm("auto")
    finite = torch.isfinite(want)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isfinite(got), finite)
    assert torch.equal(got[~finite & ~torch.isnan(want)], want[~finite & ~torch.isnan(want)])
    torch.testing.assert_close(got[finite], want[finite], rtol=1e-4, atol=1e-3)
