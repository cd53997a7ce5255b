"""Fused attention at any sequence length that is a multiple of 8 (chunks of 128 rows, blocks of 64 queries or keys, four
waves of 16; chunks of 256, blocks of 128, eight waves of 16 where there are more than 256 blocks of 64; four waves of 32
where there are more than 256 of 128) against attention in fp32 from the same bf16 operands.

Bound: P is rounded to bf16 once (2^-9 of it) and so is the result: 2-norm error below 2 x 2^-9 = 4e-3.  The backward
rounds P, dS and its results, and reads a delta formed from the rounded context: 4 x 2^-9 = 8e-3."""
import pytest
import torch

pytestmark = pytest.mark.gpu

BF = torch.bfloat16


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


def _reference(qkv, dctx, B, S, h):
    q, k, v = (t.reshape(B, S, h, 64).transpose(1, 2).float().contiguous().requires_grad_() for t in qkv.split(64 * h, 1))
    o = torch.softmax(torch.matmul(q, k.transpose(2, 3).contiguous()) / 8, -1) @ v
    o.backward(dctx.reshape(B, S, h, 64).transpose(1, 2).float().contiguous())
    back = lambda t: t.transpose(1, 2).reshape(B * S, 64 * h)
    return back(o.detach()), [back(t.grad) for t in (q, k, v)]


@pytest.mark.parametrize("late", [False, True])
@pytest.mark.parametrize("B,S,h", [(2, 8, 3), (1, 16, 2), (3, 24, 1), (2, 56, 2), (1, 64, 2), (2, 72, 3), (1, 120, 2), (2, 136, 2),
                                   (3, 200, 12), (1, 248, 1), (2, 264, 2), (1, 384, 2), (1, 520, 2), (2, 640, 2),
                                   (128, 8, 2), (64, 72, 4), (128, 120, 2), (64, 128, 4), (65, 136, 2), (43, 264, 2), (26, 520, 2),
                                   (48, 136, 2), (40, 200, 2), (128, 256, 1), (30, 264, 2), (20, 520, 2), (24, 776, 1), (43, 88, 3)])
def test_forward_and_backward(B, S, h, late):
    """``late``: the largest scores of a query lie in its last keys, so that the running maximum rises with every chunk."""
    from pipedream_amd import ops
    g = torch.Generator().manual_seed(S)
    qkv = torch.randn(B * S, 3 * 64 * h, generator=g)
    if late:
        ramp = torch.linspace(0.2, 4.0, S).repeat(B)[:, None]
        qkv[:, 64 * h:128 * h] = qkv[:, 64 * h:128 * h].abs() * ramp * 0.5
        qkv[:, :64 * h] = qkv[:, :64 * h].abs()
    qkv, dctx = qkv.to(BF).cuda(), torch.randn(B * S, 64 * h, generator=g).to(BF).cuda()
    ctx, lse2 = ops.attention_forward(qkv, B, S, h)
    assert lse2.dtype == torch.float32 and lse2.shape == (B, h, S)
    dqkv = ops.attention_backward(dctx, qkv, lse2, B, S, h, ctx=ctx)
    ref, grads = _reference(qkv, dctx, B, S, h)
    assert _rel(ctx, ref) < 4e-3
    for name, got, want in zip("qkv", dqkv.split(64 * h, 1), grads):
        # (late: nearly all weight on few keys, dS is a small difference of large numbers)
        assert _rel(got, want) < (8e-3 if not late or name == "v" else 6e-2), name


def test_rows_past_the_sequence_are_not_read_as_values():
    """Each batch entry alone gives the same bits as inside the batch (its neighbour's rows lie behind its own), and a
    NaN in one entry stays there."""
    from pipedream_amd import ops
    B, S, h = 3, 136, 2
    g = torch.Generator().manual_seed(1)
    qkv = torch.randn(B * S, 3 * 64 * h, generator=g).to(BF).cuda()
    dctx = torch.randn(B * S, 64 * h, generator=g).to(BF).cuda()
    qkv[2 * S:] = float("nan")
    ctx, lse2 = ops.attention_forward(qkv, B, S, h)
    dqkv = ops.attention_backward(dctx, qkv, lse2, B, S, h, ctx=ctx)
    for b in range(2):
        rows = slice(b * S, (b + 1) * S)
        one, l1 = ops.attention_forward(qkv[rows].contiguous(), 1, S, h)
        assert torch.equal(one, ctx[rows]) and torch.equal(l1[0], lse2[b])
        assert torch.equal(ops.attention_backward(dctx[rows].contiguous(), qkv[rows].contiguous(), l1, 1, S, h, ctx=one), dqkv[rows])
    assert torch.isnan(ctx[2 * S:].float()).all() and torch.isfinite(dqkv[:2 * S].float()).all()


@pytest.mark.parametrize("batch,heads", [(1, 2), (4, 16)])
def test_probabilities_at_512(batch, heads):
    """Written by a second pass, with blocks of 64 and of 128 queries: the context keeps its bits, a probability is one
    rounding to bf16 (half a unit in the last of 8 bits: 2^-8 at most) off, and a little for the exponential of the hardware."""
    from pipedream_amd import ops
    S, g = 512, torch.Generator().manual_seed(5)
    qkv = torch.randn(batch * S, 3 * 64 * heads, generator=g).to(BF).cuda()
    ctx, probs = ops.attention_forward(qkv, batch, S, heads, need_probs=True)
    assert torch.equal(ctx, ops.attention_forward(qkv, batch, S, heads)[0])
    q, k = (t.reshape(batch, S, heads, 64).transpose(1, 2).float().contiguous() for t in qkv.split(64 * heads, 1)[:2])
    want = torch.softmax(torch.matmul(q, k.transpose(2, 3).contiguous()) / 8, -1)
    assert float(((probs.float() - want).abs() / want).max()) < 2.0 ** -8 + 1e-4


@pytest.mark.parametrize("B,S,h", [(1, 200, 2), (2, 512, 2), (1, 264, 1), (8, 512, 8), (43, 264, 2), (30, 264, 2)])
def test_scores_that_are_infinite(B, S, h):
    """Query 0: the first 128 keys at -inf (finite operands whose products overflow), finite ones after them.  Query 1: all
    but the last key.  Query 2: every key at -inf, query 3: one at +inf, both NaN as in fp32.  The others are ordinary."""
    from pipedream_amd import ops
    g = torch.Generator().manual_seed(S + 1)
    qkv, dctx = torch.randn(B * S, 3 * 64 * h, generator=g), torch.randn(B * S, 64 * h, generator=g)
    q, k, _ = (t.view(B, S, h, 64) for t in qkv.split(64 * h, 1))
    q[..., :4], k[..., :4] = 0.0, 0.0
    for i in range(4):
        q[:, i, :, i] = 1e30
    k[:, :128, :, 0] = -1e30
    k[:, :S - 1, :, 1] = -1e30
    k[:, :, :, 2] = -1e30
    k[:, 150, :, 3] = 1e30
    qkv, dctx = qkv.to(BF).cuda(), dctx.to(BF).cuda()
    ctx, lse2 = ops.attention_forward(qkv, B, S, h)
    ref, grads = _reference(qkv.cpu(), dctx.cpu(), B, S, h)
    got, want = ctx.cpu().view(B, S, -1), ref.view(B, S, -1)
    ordinary = [0, 1] + list(range(4, S))
    assert torch.isnan(want[:, 2:4]).all() and torch.isnan(got[:, 2:4].float()).all()
    assert torch.isfinite(want[:, ordinary]).all() and _rel(got[:, ordinary], want[:, ordinary]) < 4e-3
    for i in (0, 1):
        assert _rel(got[:, i], want[:, i]) < 8e-3          # (one row: a rounding of P and one of the result each)
    # the gradients of the queries, without the NaNs that reach every key from queries 2 and 3
    dq = ops.attention_backward(dctx, qkv, lse2, B, S, h, ctx=ctx)[:, :64 * h].cpu().view(B, S, -1)
    want = grads[0].view(B, S, -1)
    rows = list(range(4, S))
    cols = [64 * i + j for i in range(h) for j in range(4, 64)]        # (the first four columns of K hold the 1e30)
    assert _rel(dq[:, rows][..., cols], want[:, rows][..., cols]) < 8e-3


@pytest.mark.parametrize("S", [8, 200, 264])
def test_backward_without_the_context(S):
    from pipedream_amd import ops
    g = torch.Generator().manual_seed(S)
    qkv, dctx = torch.randn(2 * S, 3 * 128, generator=g).to(BF).cuda(), torch.randn(2 * S, 128, generator=g).to(BF).cuda()
    ctx, aux = ops.attention_forward(qkv, 2, S, 2)
    assert torch.equal(ops.attention_backward(dctx, qkv, aux, 2, S, 2), ops.attention_backward(dctx, qkv, aux, 2, S, 2, ctx=ctx))
    with pytest.raises(ValueError):
        ops.attention_backward(dctx, qkv, aux, 2, S, 2, ctx=ctx[:S])


def test_lengths_that_always_needed_the_context_still_do():
    from pipedream_amd import ops
    qkv = torch.randn(128, 3 * 64).to(BF).cuda()
    ctx, aux = ops.attention_forward(qkv, 1, 128, 1)
    with pytest.raises(ValueError):
        ops.attention_backward(torch.ones_like(ctx), qkv, aux, 1, 128, 1)
