"""Which parameters the native calls of a transformer layer take: they see pointers alone, so every shape is compared before
one is handed over, and what the single launches do not compare themselves is refused."""
import types

import pytest
import torch

from pipedream_amd import layers, ops


def _params(hidden=64, ffn=96, **other):
    layer = layers.TransformerLayer(hidden, 1, ffn)
    for name, module in other.items():
        setattr(layer, name, module)
    return tuple(p for m in (layer.ln1, layer.qkv, layer.proj, layer.ln2, layer.fc1, layer.fc2) for p in (m.weight, m.bias))


def test_the_layers_own_parameters_fit():
    assert ops._layer_fits(_params(), 64)
    ops.check_layer_vectors(_params(), 64)


@pytest.mark.parametrize("features", [32, 63, 72, 128])
def test_another_number_of_features_does_not_fit(features):
    assert not ops._layer_fits(_params(), features)


LINEAR, NORM = torch.nn.Linear, torch.nn.LayerNorm


@pytest.mark.parametrize("name,module", [("ln1", NORM(72)), ("ln1", NORM(56)), ("ln2", NORM(128)), ("qkv", LINEAR(64, 200)),
                                         ("qkv", LINEAR(72, 192)), ("qkv", LINEAR(64, 96)), ("proj", LINEAR(64, 72)),
                                         ("proj", LINEAR(32, 64)), ("fc1", LINEAR(64, 128)), ("fc1", LINEAR(72, 96)),
                                         ("fc2", LINEAR(128, 64)), ("fc2", LINEAR(96, 72)), ("fc2", LINEAR(96, 64, bias=False))])
def test_a_replaced_module_does_not_fit(name, module):
    assert not ops._layer_fits(_params(**{name: module}), 64)


@pytest.mark.parametrize("place", range(12))
def test_a_parameter_that_is_too_short_is_refused(place):
    params = list(_params())
    params[place] = torch.nn.Parameter(params[place].detach()[:-8].clone())
    assert not ops._layer_fits(params, 64)
    if place in (0, 1, 3, 5, 6, 7, 9, 11):
        with pytest.raises(ValueError):
            ops.check_layer_vectors(params, 64)


@pytest.mark.parametrize("B,S,hidden,heads,ffn", [(2, 16, 64, 1, 96), (3, 200, 768, 12, 3072), (1, 8, 64, 2, 8), (2, 24, 96, 3, 104)])
def test_the_tensors_a_forward_pass_leaves_lie_side_by_side(B, S, hidden, heads, ffn):
    """Every tensor on a 256-byte boundary, in order, none over another, the last one inside the buffer."""
    saved = torch.zeros(ops._layer_bytes(B, S, heads, hidden, ffn)[0], dtype=torch.uint8)
    at = 0
    for t in ops.transformer_layer_saved(saved, B, S, heads, hidden, ffn):
        start = t.data_ptr() - saved.data_ptr()
        assert start % 256 == 0 and at <= start < at + 256
        at = start + t.numel() * t.element_size()
    assert at <= saved.numel() < at + 256


@pytest.mark.gpu
@pytest.mark.parametrize("timer", [None, {}])
@pytest.mark.parametrize("built,given", [(128, 256), (256, 128)])
def test_a_layer_for_other_features_raises(built, given, timer):
    layer = layers.TransformerLayer(built, built // 64, 2 * built).cuda()
    x = torch.zeros(2, 16, given, dtype=torch.bfloat16, device="cuda")
    ops.kernel_timer = timer
    try:
        with pytest.raises(ValueError):
            layer(x)
    finally:
        ops.kernel_timer = None


@pytest.mark.gpu
@pytest.mark.parametrize("name,rows,cols", [("fc1", 320, 128), ("fc1", 256, 64), ("fc2", 128, 320), ("proj", 128, 64), ("qkv", 192, 128)])
def test_a_replaced_linear_raises_in_either_pass(name, rows, cols):
    layer = layers.TransformerLayer(128, 2, 256).cuda()
    x = torch.randn(2, 16, 128).bfloat16().cuda().requires_grad_()
    y = layer(x)
    kept = getattr(layer, name)
    other = torch.nn.Linear(cols, rows).cuda()
    with pytest.raises(ValueError):
        setattr(layer, name, other)
        layer(x)
    setattr(layer, name, kept)
    kept.weight.data, kept.bias.data = other.weight.data, other.bias.data       # between the passes
    with pytest.raises((ValueError, RuntimeError)):
        y.backward(torch.ones_like(y))


@pytest.mark.gpu
def test_a_bf16_image_of_another_shape_raises():
    """The image that an optimizer keeps of a weight is what the kernels read: one of fewer rows than the weight, from before its
    data was replaced."""
    layer = layers.TransformerLayer(128, 2, 256).cuda()
    layer.fc2.weight._pd_arena = types.SimpleNamespace(live_slot=0)
    layer.fc2.weight._pd_bf16_views = [torch.zeros(64, 256, dtype=torch.bfloat16, device="cuda")]
    with pytest.raises(ValueError):
        layer(torch.zeros(2, 16, 128, dtype=torch.bfloat16, device="cuda"))


@pytest.mark.gpu
def test_layers_without_a_bias_or_with_another_attention_width_run():
    """What the single launches take: a forward pass without biases, attention of 64 features (two heads of 32) in a layer of
    128."""
    g = torch.Generator().manual_seed(4)
    x = torch.randn(2, 16, 128, generator=g).bfloat16().cuda()
    layer = layers.TransformerLayer(128, 2, 256).cuda()
    with torch.no_grad():
        for m in (layer.qkv, layer.proj, layer.fc1, layer.fc2):
            m.bias.zero_()
        want = layer(x)
        for m in (layer.qkv, layer.proj, layer.fc1, layer.fc2):
            m.bias = None
        assert torch.equal(layer(x), want)
    layer = layers.TransformerLayer(128, 2, 256)
    layer.qkv, layer.proj = torch.nn.Linear(128, 192), torch.nn.Linear(64, 128)
    layer = layer.cuda()
    xr = x.clone().requires_grad_()
    y = layer(xr)
    y.backward(torch.ones_like(y))
    assert torch.isfinite(y.float()).all() and torch.isfinite(xr.grad.float()).all()
    assert layer.qkv.weight.grad.shape == (192, 128) and layer.proj.weight.grad.shape == (128, 64)
