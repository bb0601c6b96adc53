"""The residual stream's sum, and the sum of its gradients, inside the norm's kernels."""

import pytest
import torch

from automodel_amd.ops.rms_norm import RMSNorm, add_norm

gpu = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def f64(x, delta, w, eps, g_sum, g_y):
    x, delta, w = (None if t is None else t.detach().double().requires_grad_() for t in (x, delta, w))
    # the sum is rounded to bf16 before it is normed
    s = x if delta is None else x + delta
    s = s + (s.bfloat16().double() - s).detach()
    y = s * torch.rsqrt((s * s).mean(-1, keepdim=True) + eps) * w
    grads = torch.autograd.grad((s, y), [x, w], (g_sum.double(), g_y.double()))
    return s, y, *grads


@pytest.mark.parametrize("T,H", [(1, 8), (67, 136), (300, 512), (2051, 2048), (5, 2056), (1100, 4096),
                                 (2, 16384)])
@pytest.mark.parametrize("with_delta", [False, True])
@pytest.mark.parametrize("frozen", [False, True])
@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")
def test_kernels(T, H, with_delta, frozen):
    torch.manual_seed(0)
    norm = RMSNorm(H, 1e-5, device="cuda", dtype=torch.bfloat16)
    with torch.no_grad():
        norm.weight += 0.1 * torch.randn_like(norm.weight)
    norm.weight.requires_grad_(not frozen)
    x, delta, g_sum, g_y = (torch.randn(T, H, device="cuda").bfloat16() for _ in range(4))
    x.requires_grad_()
    delta = delta.requires_grad_() if with_delta else None
    s, y = add_norm(norm, x, delta)
    assert "AddRMSNorm" in y.grad_fn.name()
    torch.autograd.backward((s, y), (g_sum, g_y))
    rs, ry, gx, gw = f64(x, delta, norm.weight, 1e-5, g_sum, g_y)
    assert torch.equal(s.double(), rs)
    # y is rounded before and after the weight, gradients once
    for got, want, roundings in ((y, ry, 2), (x.grad, gx, 1), (norm.weight.grad, gw, 1)):
        if got is not None:
            assert (got.double() - want).norm() <= roundings * 2.0 ** -9 * want.norm() + 1e-12
    assert (norm.weight.grad is None) == frozen
    if with_delta:
        assert torch.equal(delta.grad, x.grad)


@pytest.mark.parametrize("device", ["cpu", pytest.param("cuda", marks=gpu)])
def test_either_output_alone_and_other_calls(device):
    """One output's gradient, hooks, other types and strides: as the module by itself."""
    dtype = torch.bfloat16 if device == "cuda" else torch.float32
    torch.manual_seed(0)
    norm = RMSNorm(64, 1e-5, device=device, dtype=dtype)
    base, delta = (torch.randn(4, 6, 64, device=device, dtype=dtype) for _ in range(2))
    for make in (lambda t: t, lambda t: t.transpose(0, 1), lambda t: t[:, :1].expand(4, 6, 64),
                 lambda t: t.float()):
        x, d = make(base).detach().requires_grad_(), make(delta).detach().requires_grad_()
        if x.dtype != dtype:
            norm = norm.float()
            if device == "cuda":
                continue                      # the kernels take bf16 only
        for which in (0, 1):
            got = torch.autograd.grad(add_norm(norm, x, d)[which].sum(), (x, d))
            s = x + d
            want = torch.autograd.grad((s, norm(s))[which].sum(), (x, d))
            for a, b in zip(got, want):
                torch.testing.assert_close(a, b, atol=2e-2, rtol=2e-2)
    norm = RMSNorm(64, 1e-5, device=device, dtype=dtype)
    seen = []
    norm.register_forward_hook(lambda m, i, o: seen.append(o))
    s, y = add_norm(norm, base, delta)
    assert len(seen) == 1 and y is seen[0]
