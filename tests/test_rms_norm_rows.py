"""RMSNorm kernels over all kinds of row lengths (part of a wave, a wave, a workgroup)."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("T,H", [(1, 8), (5, 128), (67, 136), (9, 256), (300, 512), (33, 520), (7, 1024),
                                 (1, 520), (96, 768), (97, 768), (769, 768), (64, 2048), (256, 2048), (2040, 2040),
                                 (2051, 2048), (5, 2056), (1100, 4096), (3, 8192), (2, 16384)])
def test_forward_backward(T, H):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    x, dy = (torch.randn(T, H, device="cuda").bfloat16() for _ in range(2))
    w = (1 + 0.1 * torch.randn(H, device="cuda")).bfloat16()
    y, inv = hip_ops().rms_norm_fwd(x, w, 1e-5)
    dx, dw = hip_ops().rms_norm_bwd(dy, x, w, inv)
    xd, wd = x.double().requires_grad_(), w.double().requires_grad_()
    r = torch.rsqrt((xd * xd).mean(-1, keepdim=True) + 1e-5)
    ref = xd * r * wd
    gx, gw = torch.autograd.grad(ref, (xd, wd), dy.double())
    # y: rounded to bf16 before and after the weight; gradients once
    for got, want, roundings in ((y, ref, 2), (dx, gx, 1), (dw, gw, 1)):
        assert (got.double() - want).norm() <= roundings * 2.0 ** -9 * want.norm() + 1e-12
    again = hip_ops().rms_norm_bwd(dy, x, w, inv)
    assert torch.equal(again[1], dw)            # the sums have a fixed order


def test_forward_long_rows():
    from automodel_amd.ops._backend import hip_ops

    x = torch.randn(3, 20000, device="cuda").bfloat16()
    w = torch.ones(20000, device="cuda").bfloat16()
    y, _ = hip_ops().rms_norm_fwd(x, w, 1e-5)
    ref = x.double() * torch.rsqrt((x.double() ** 2).mean(-1, keepdim=True) + 1e-5)
    assert (y.double() - ref).norm() <= 2.0 ** -8 * ref.norm()
