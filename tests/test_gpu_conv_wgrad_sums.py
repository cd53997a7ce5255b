"""The sums over the blocks' partial weight gradients (pd_conv3x3_winograd.hip) for every number of block pairs: 4 to 64
ranks added up to one before the final kernel, or all of them in it; a weight gradient that is not 16-byte aligned.

Bound: as for the kernels that write the partials (2.5e-6 of the gradient in the 2-norm is above what any of them shows);
the bias gradient adds N H W values in fp32, pairwise: 1e-6."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

CL = torch.channels_last


def _operands(N, C, K, H, W):
    g = torch.Generator().manual_seed(C + K)
    x = torch.randn(N, C, H, W, generator=g).cuda().contiguous(memory_format=CL)
    dy = torch.randn(N, K, H, W, generator=g).cuda().contiguous(memory_format=CL)
    return x, dy


@pytest.mark.parametrize("N,H,W", [(2, 18, 14), (8, 33, 30)])
@pytest.mark.parametrize("C,K", [(64, 64), (128, 64), (128, 128), (128, 256), (256, 256), (512, 256), (512, 512), (1024, 1024)])
def test_weight_gradient_matches_64_bits(N, H, W, C, K):
    from pipedream_amd import _cabi, ops
    assert _cabi.lib().pd_conv3x3_winograd_wgrad_supported(C, K)
    x, dy = _operands(N, C, K, H, W)
    dw, db = ops.conv3x3_weight_grad(x, dy)
    ref = torch.nn.grad.conv2d_weight(x.cpu().double(), (K, C, 3, 3), dy.cpu().double(), padding=1) if C <= 256 else None
    if ref is not None:
        assert float((dw.cpu().double() - ref).norm() / ref.norm()) < 2.5e-6
    else:                                          # (one tap by a product: the whole reference takes half a minute)
        a = torch.nn.functional.pad(x, (1, 1, 1, 1)).double()[:, :, 0:H, 2:2 + W].permute(1, 0, 2, 3).reshape(C, -1)
        tap = dy.double().permute(1, 0, 2, 3).reshape(K, -1) @ a.t().contiguous()
        assert float((dw[:, :, 0, 2].double() - tap).norm() / tap.norm()) < 2.5e-6
    dbr = dy.double().sum((0, 2, 3))
    assert float((db.double() - dbr).norm() / dbr.norm()) < 1e-6
    again, _ = ops.conv3x3_weight_grad(x, dy)
    assert torch.equal(dw, again)


def test_unaligned_result():
    from pipedream_amd import _cabi, ops
    x, dy = _operands(2, 64, 64, 18, 14)
    want, _ = ops.conv3x3_weight_grad(x, dy)
    lib, nbytes = _cabi.lib(), ctypes.c_uint64()
    lib.pd_conv3x3_winograd_wgrad_workspace_bytes(64, 64, ctypes.byref(nbytes))
    ws = torch.empty(nbytes.value, dtype=torch.uint8, device="cuda")
    flat = torch.zeros(64 * 9 * 64 + 2, device="cuda")
    lib.pd_conv3x3_winograd_wgrad_nhwc_f32(x.data_ptr(), dy.data_ptr(), flat[1:].data_ptr(), None, ws.data_ptr(), nbytes.value,
                                           2, 18, 14, 64, 64, _cabi.stream_ptr())
    assert torch.equal(flat[1:-1].view(64, 3, 3, 64).permute(0, 3, 1, 2), want) and not flat[0] and not flat[-1]
