"""A transformer layer's passes as one native call each against the same launches issued one by one (the path of the
per-launch timer): the same bits, whichever of the two a pass takes, for fused and unfused attention, token counts that
split the weight gradients and ones that do not, fresh gradients and accumulated ones."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _layer(hidden, heads, ffn):
    from pipedream_amd import layers
    torch.manual_seed(1)
    layer = layers.TransformerLayer(hidden, heads, ffn)
    for p in layer.parameters():
        if p.dim() == 1:
            torch.nn.init.normal_(p, 0.5 if p is layer.ln1.weight or p is layer.ln2.weight else 0.0, 0.2)
    return layer.cuda()


def _passes(layer, xs, dys, forward_native, backward_native):
    from pipedream_amd import ops
    for p in layer.parameters():
        p.grad = None
    out = []
    try:
        for x, dy in zip(xs, dys):
            x = x.detach().requires_grad_()
            ops.kernel_timer = None if forward_native else {}
            y = layer(x)
            ops.kernel_timer = None if backward_native else {}
            y.backward(dy)
            out += [y.detach(), x.grad]
    finally:
        ops.kernel_timer = None
    return out + [p.grad for p in layer.parameters()]


@pytest.mark.parametrize("B,S,hidden,heads,ffn", [(2, 64, 128, 4, 256), (1, 40, 128, 2, 512), (3, 128, 192, 3, 256),
                                                  (1, 8, 64, 1, 64), (4, 512, 256, 4, 512), (2, 200, 128, 2, 384)])
def test_native_passes_equal_the_single_launches(B, S, hidden, heads, ffn):
    layer = _layer(hidden, heads, ffn)
    g = torch.Generator().manual_seed(2)
    xs = [torch.randn(B, S, hidden, generator=g).bfloat16().cuda() for _ in range(2)]
    dys = [(torch.randn(B, S, hidden, generator=g) * 0.1).bfloat16().cuda() for _ in range(2)]
    want = _passes(layer, xs, dys, False, False)
    for forward_native, backward_native in ((True, True), (True, False), (False, True)):
        for a, b in zip(_passes(layer, xs, dys, forward_native, backward_native), want):
            assert torch.equal(a, b)


def test_gradients_that_are_not_dense_take_the_single_launches():
    layer = _layer(64, 1, 64)
    x, dy = torch.randn(1, 16, 64).bfloat16().cuda(), torch.randn(1, 16, 64).bfloat16().cuda()
    want = _passes(layer, [x], [dy], True, True)
    layer.zero_grad(set_to_none=True)
    wide = torch.zeros(64, 128).cuda()
    layer.proj.weight.grad = wide[:, :64]
    layer(x.requires_grad_()).backward(dy)
    for p, w in zip(layer.parameters(), want[2:]):
        assert torch.equal(p.grad, w)
    assert layer.proj.weight.grad.data_ptr() == wide.data_ptr() and not wide[:, 64:].any()


def test_weights_read_by_the_backward_pass_are_the_current_ones():
    """The backward pass reads the parameters when it runs (weight stashing swaps them in between)."""
    layer = _layer(64, 1, 64)
    x, dy = torch.randn(1, 16, 64).bfloat16().cuda(), torch.randn(1, 16, 64).bfloat16().cuda()
    xs = []
    for change in (False, True):
        xi = x.detach().requires_grad_()
        y = layer(xi)
        if change:
            layer.fc2.weight.data.mul_(2.0)
        y.backward(dy)
        xs.append(xi.grad)
    assert not torch.equal(xs[0], xs[1])


def test_one_matrix_in_two_places_gets_both_gradients():
    """fc1 and fc2 as one parameter: what separate copies get, added up, in a first pass and in an accumulated one."""
    layer = _layer(64, 1, 64)
    g = torch.Generator().manual_seed(3)
    x, dy = (torch.randn(2, 16, 64, generator=g).bfloat16().cuda() for _ in range(2))
    layer.fc2.weight.data = layer.fc1.weight.data.clone()
    _passes(layer, [x, x], [dy, dy], True, True)
    want = layer.fc1.weight.grad.double() + layer.fc2.weight.grad.double()
    others = [p.grad.clone() for p in layer.parameters() if p is not layer.fc1.weight and p is not layer.fc2.weight]
    layer.fc2.weight = layer.fc1.weight
    _passes(layer, [x, x], [dy, dy], True, True)
    assert float((layer.fc1.weight.grad.double() - want).norm() / want.norm()) < 1e-6
    for a, b in zip([p.grad for p in layer.parameters() if p is not layer.fc1.weight], others):
        assert torch.equal(a, b)


def test_saved_tensors_may_come_back_at_another_address():
    """Hooks that keep what the forward pass saved in a buffer of their own, on boundaries of 16 bytes only."""
    layer = _layer(64, 1, 64)
    x, dy = torch.randn(2, 16, 64).bfloat16().cuda(), torch.randn(2, 16, 64).bfloat16().cuda()
    want = _passes(layer, [x], [dy], True, True)

    def elsewhere(t):
        n = t.numel() * t.element_size()
        buf = torch.empty(n + 16, dtype=torch.uint8, device=t.device)[16:]
        buf.copy_(t.reshape(-1).view(torch.uint8))
        return buf.view(t.dtype).view(t.shape)

    with torch.autograd.graph.saved_tensors_hooks(elsewhere, lambda t: t):
        got = _passes(layer, [x], [dy], True, True)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("B,S", [(2, 16), (4, 512)])
@pytest.mark.parametrize("name,shape", [("fc2.weight", (64, 32)), ("fc1.weight", (128, 64)), ("qkv.bias", (64,)),
                                        ("ln1.weight", (72,))])
def test_a_gradient_of_another_shape_raises(B, S, name, shape):
    """A parameter whose data had another shape when its gradient was made: the kernels would write past the gradient's end."""
    layer = _layer(64, 1, 64)
    p = layer.get_parameter(name)
    kept = p.data
    p.data = torch.zeros(shape, device="cuda")
    p.grad = torch.zeros(shape, device="cuda")
    p.data = kept
    y = layer(torch.randn(B, S, 64).bfloat16().cuda().requires_grad_())
    with pytest.raises((ValueError, RuntimeError)):
        y.backward(torch.ones_like(y))
