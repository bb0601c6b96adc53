"""RMSNorm with a CDNA4 HIP kernel (fwd+bwd) and a torch reference path.

Replaces the reference's TE/QuACK/Liger RMSNorm backends
(nemo_automodel/components/models/common/utils.py:282, kernel_patches.py:155)
with one hand-written HIP kernel (csrc/rms_norm.hip).
"""

from __future__ import annotations

import torch

from automodel_amd.ops._backend import hip_ops


def rms_norm_ref(x: torch.Tensor, weight: torch.Tensor, eps: float) -> torch.Tensor:
    """fp32-upcast reference (used on CPU and in kernel parity tests)."""
    xf = x.float()
    inv = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
    return (xf * inv).to(x.dtype) * weight


class _RMSNormHip(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x: torch.Tensor, weight: torch.Tensor, eps: float):
        x2d = x.reshape(-1, x.shape[-1]).contiguous()
        y, invrms = hip_ops().rms_norm_fwd(x2d, weight, eps)
        ctx.save_for_backward(x2d, weight, invrms)
        ctx.x_shape = x.shape
        return y.view(x.shape)

    @staticmethod
    def backward(ctx, dy: torch.Tensor):
        x2d, weight, invrms = ctx.saved_tensors
        dy2d = dy.reshape(-1, dy.shape[-1]).contiguous()
        want_dw = ctx.needs_input_grad[1]
        dx, dw = hip_ops().rms_norm_bwd(dy2d, x2d, weight, invrms, None, want_dw)
        return dx.view(ctx.x_shape), dw.to(weight.dtype) if want_dw else None, None


class _AddRMSNormHip(torch.autograd.Function):
    """(x, delta) -> x + delta and its norm; without delta x itself and its norm. The two
    gradients of the stream are added in the norm's backward."""

    @staticmethod
    def forward(ctx, x: torch.Tensor, delta: torch.Tensor | None, weight: torch.Tensor, eps: float):
        x2d = x.reshape(-1, x.shape[-1]).contiguous()
        if delta is None:
            total = x
            y, invrms = hip_ops().rms_norm_fwd(x2d, weight, eps)
        else:
            x2d, y, invrms = hip_ops().add_rms_norm_fwd(
                x2d, delta.reshape(x2d.shape).contiguous(), weight, eps)
            total = x2d.view(x.shape)
        ctx.save_for_backward(x2d, weight, invrms)
        ctx.set_materialize_grads(False)
        return total, y.view(x.shape)

    @staticmethod
    def backward(ctx, dtotal: torch.Tensor | None, dy: torch.Tensor | None):
        x2d, weight, invrms = ctx.saved_tensors
        dw = None
        dx = dtotal
        if dy is not None:
            want_dw = ctx.needs_input_grad[2]
            shape, dy = dy.shape, dy.reshape(x2d.shape).contiguous()
            if dtotal is not None:
                dtotal = dtotal.reshape(x2d.shape).contiguous()
            dx, dw = hip_ops().rms_norm_bwd(dy, x2d, weight, invrms, dtotal, want_dw)
            dx = dx.view(shape)
        return dx, dx if ctx.needs_input_grad[1] else None, dw, None


def rms_norm(x: torch.Tensor, weight: torch.Tensor, eps: float = 1e-6, backend: str = "hip") -> torch.Tensor:
    if backend == "hip" and x.is_cuda:
        return _RMSNormHip.apply(x, weight, eps)
    return rms_norm_ref(x, weight, eps)


def add_norm(norm: torch.nn.Module, x: torch.Tensor,
             delta: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor]:
    """``s = x + delta`` (x without delta) and ``norm(s)``, for a residual stream that goes
    on from s: in one pass where the kernel applies, whose backward also adds up the two
    gradients of s."""
    w = getattr(norm, "weight", None)
    hooks = torch.nn.modules.module
    if (type(norm) is RMSNorm and norm.backend == "hip" and x.is_cuda
            and type(x) is torch.Tensor and x.dtype == torch.bfloat16 and x.numel()
            and (delta is None or (type(delta) is torch.Tensor and delta.shape == x.shape
                                   and delta.dtype == x.dtype and delta.device == x.device))
            and type(w) in (torch.nn.Parameter, torch.Tensor) and w.dtype == x.dtype
            and w.shape == x.shape[-1:] and w.is_contiguous() and w.device == x.device
            and x.shape[-1] % 8 == 0 and x.shape[-1] <= 16384
            and not (norm._forward_hooks or norm._forward_pre_hooks or norm._backward_hooks
                     or norm._backward_pre_hooks or hooks._global_forward_hooks
                     or hooks._global_forward_pre_hooks or hooks._global_backward_hooks
                     or hooks._global_backward_pre_hooks)):
        return _AddRMSNormHip.apply(x, delta, w, norm.variance_epsilon)
    s = x if delta is None else x + delta
    return s, norm(s)


class RMSNorm(torch.nn.Module):
    def __init__(self, hidden_size: int, eps: float = 1e-6, backend: str = "hip",
                 device=None, dtype=None):
        super().__init__()
        self.weight = torch.nn.Parameter(torch.ones(hidden_size, device=device, dtype=dtype))
        self.variance_epsilon = eps
        self.backend = backend

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return rms_norm(x, self.weight, self.variance_epsilon, self.backend)

    def reset_parameters(self) -> None:
        torch.nn.init.ones_(self.weight)

    def extra_repr(self) -> str:
        return f"{self.weight.shape[0]}, eps={self.variance_epsilon}, backend={self.backend}"
