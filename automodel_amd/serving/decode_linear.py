"""Decode-path linear layers on the kernels of ops/csrc/gemv.hip.

Reference behavior: serving engines (which the reference defers to for
deployment) special-case decode GEMVs; here the kernels are in-tree.
``decode_rows`` is what cached decoding of the Llama family calls,
``project`` the packed rows of the models with slot caches, and DecodeLinear
swaps in for inference. Training paths are untouched: the kernels only run
under no_grad with few bf16 rows on the GPU; everything else falls through
to F.linear (hipBLASLt)."""

from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F

from automodel_amd.ops.linear import gated, inferred, squared_own

_PAD_TO = {5: 8, 6: 8, 7: 8, 9: 16, 10: 16, 11: 16, 12: 16, 13: 16, 14: 16, 15: 16}


def gemv_bf16(x2d: torch.Tensor, w: torch.Tensor, bias: torch.Tensor | None = None,
              relu2: bool = False, out_f32: bool = False) -> torch.Tensor:
    """y = x2d @ w.T via the HIP kernel; pads odd batch sizes to a
    compiled template instance. Epilogues: max(y, 0)^2, f32 output."""
    from automodel_amd.ops._backend import hip_ops

    B = x2d.shape[0]
    tgt = _PAD_TO.get(B, B)
    if tgt != B:
        x2d = F.pad(x2d, (0, 0, 0, tgt - B))
    y = hip_ops().gemv_bf16(x2d, w, bias, relu2, out_f32)
    return y[:B] if tgt != B else y


def _gemv_eligible(x: torch.Tensor, w: torch.Tensor) -> bool:
    if torch.is_grad_enabled() or not x.is_cuda:
        return False
    if x.dtype != torch.bfloat16 or w.dtype != torch.bfloat16:
        return False
    rows = x.numel() // x.shape[-1]
    # measured on MI355X (profiles/README.md): the wave-per-row GEMV beats
    # hipBLASLt up to ~4 rows; above that `inferred` chooses
    return rows <= 4 and x.shape[-1] % 512 == 0


def project(lin: nn.Module, x: torch.Tensor, relu2: bool = False,
            out_f32: bool = False) -> torch.Tensor:
    """``lin(x)`` for packed rows x [T, K], optionally followed by max(y, 0)^2
    and optionally in float32 (a residual input or logits must not be rounded
    to bf16 on the way out of the accumulator).

    Inference on the GPU: up to 2 bf16 rows take the GEMV, up to 64 the skinny
    MFMA GEMM, both with fused epilogues; more take the faster one of the kernels of
    ops/linear.py and the library's GEMM. Wrapped layers (adapters) and autograd take the
    module itself."""
    from automodel_amd.ops import residual_norm as rn

    if type(lin) not in (nn.Linear, DecodeLinear) or lin.bias is not None or not rn.use_hip(x):
        y = lin(x)
        y = rn.relu2(y) if relu2 else y
        return y.float() if out_f32 else y
    w = lin.weight
    if x.shape[0] == 0:
        return x.new_empty(0, w.shape[0], dtype=torch.float32 if out_f32 else x.dtype)
    if x.dtype == torch.bfloat16 and x.shape[0] <= 64 and x.shape[1] % 8 == 0:
        if x.shape[0] <= 2:
            return gemv_bf16(x, w, None, relu2, out_f32)
        from automodel_amd.ops._backend import hip_ops

        return hip_ops().gemm_skinny_bf16(x, w, relu2, out_f32)
    if out_f32 and x.dtype == torch.bfloat16:
        y = torch.mm(x, w.t(), out_dtype=torch.float32)
    else:
        squared = relu2 and squared_own(x.shape[0], *w.shape)
        y = inferred(x, w, squared)
        if squared and y is not None:
            return y
        y = F.linear(x, w) if y is None else y
    return rn.relu2(y) if relu2 else y


def project_grouped(lin: nn.Module, xs: torch.Tensor, sizes: list[int]) -> list[torch.Tensor]:
    """Several inputs through one stacked projection: the weight's rows, split by
    ``sizes``, apply to xs[i] each, xs [n, T, K]. -> the n outputs [T, sizes[i]].

    Up to 64 bf16 rows on the GPU are one launch (the outputs are slices of one
    [T, N] tensor then, see ``grouped_rows``); more take a GEMM each. A wrapped
    layer (adapters) sees every input as a whole."""
    y = grouped_rows(lin, xs, sizes)
    if y is not None:
        return list(y.split(sizes, dim=1))
    if type(lin) not in (nn.Linear, DecodeLinear):
        return [lin(x).split(sizes, dim=-1)[i] for i, x in enumerate(xs)]
    return [F.linear(x, w) for x, w in zip(xs, lin.weight.split(sizes))]


def grouped_rows(lin: nn.Module, xs: torch.Tensor, sizes: list[int]) -> torch.Tensor | None:
    """The one-launch form of ``project_grouped``, [T, N], if it applies: equal
    sizes, of which the last may be smaller."""
    from automodel_amd.ops import residual_norm as rn

    n, T, K = xs.shape
    group = sizes[0]
    if not (rn.use_hip(xs) and xs.dtype == torch.bfloat16 and 1 <= T <= 64 and K % 8 == 0
            and type(lin) in (nn.Linear, DecodeLinear) and lin.bias is None
            and sizes[:-1] == [group] * (n - 1) and 1 <= sizes[-1] <= group
            and group % (2 if T <= 4 else 16) == 0):
        return None
    w = lin.weight
    from automodel_amd.ops._backend import hip_ops

    x = xs.reshape(n * T, K)
    if T <= 2 or group % 16:
        return hip_ops().gemv_bf16(x, w, None, False, False, group)
    return hip_ops().gemm_skinny_bf16(x, w, False, False, group)


def unobserved(*modules: nn.Module) -> bool:
    """No hook would see these modules' calls, so that kernels may take their place."""
    every = nn.modules.module
    if every._global_forward_hooks or every._global_forward_pre_hooks:
        return False
    return not any(m._forward_hooks or m._forward_pre_hooks for m in modules)


def plain_linears(*lins: nn.Module) -> bool:
    """Each call is x W^T and nothing else: no adapter, no bias, no hook of a wrapper or an
    observer, no sharded weight."""
    return unobserved(*lins) and all(
        type(lin) in (nn.Linear, DecodeLinear) and lin.bias is None
        and type(lin.weight) in (nn.Parameter, torch.Tensor) for lin in lins)


def plain_weights(*lins: nn.Module) -> list[torch.Tensor] | None:
    """The weights of ``lins`` if they are ``plain_linears``. (From the modules' own tables: a module's
    ``__getattr__`` is 0.2 us, and a decode step asks some hundred times.)"""
    every = nn.modules.module
    if every._global_forward_hooks or every._global_forward_pre_hooks:
        return None
    ws = []
    for lin in lins:
        own = lin.__dict__
        if type(lin) not in (nn.Linear, DecodeLinear) or own["_forward_hooks"] or own["_forward_pre_hooks"]:
            return None
        params = own["_parameters"]
        w = params["weight"] if "weight" in params else lin.weight
        if (type(w) not in (nn.Parameter, torch.Tensor)
                or (params["bias"] if "bias" in params else lin.bias) is not None):
            return None
        ws.append(w)
    return ws


def decode_rows(lins: list[nn.Module], x: torch.Tensor,
                glu: bool = False) -> list[torch.Tensor] | None:
    """``[lin(x) for lin in lins]`` in one launch, up to three layers; with ``glu``
    ``[silu(a) * b]`` of the two outputs a and b, or of the halves of one layer's.
    None where the kernels don't apply, and nothing is done.

    Up to 32 rows: with them the library is as fast on wide layers and slower on narrow
    ones (32 rows, 14336 x 4096 26.0 us against 26.4, 8192 x 8192 30.8 and 28.4, 1024 x
    4096 11.8 and 9.3; only 10240 x 8192 stands out, 38 and 48), with more it is faster on
    most (48 rows, 14336 x 4096 28.3 and 36.2, 4096 x 4096 13.7 and 16.6)."""
    K = x.shape[-1]
    rows = x.numel() // max(K, 1)
    if not (x.is_cuda and x.dtype == torch.bfloat16 and 1 <= rows <= 32 and K % 8 == 0
            and not torch.is_grad_enabled() and not torch.is_autocast_enabled("cuda")
            and type(x) is torch.Tensor and x.is_contiguous() and x.data_ptr() % 16 == 0
            and plain_linears(*lins)):
        return None
    ws = [lin.weight for lin in lins]
    if glu and len(ws) == 1:
        ws = list(ws[0].chunk(2))
    if not all(w.dtype == torch.bfloat16 and w.is_contiguous() and w.device == x.device
               and w.data_ptr() % 16 == 0 for w in ws):
        return None
    if glu and rows * ws[0].shape[0] % 8:         # the activation kernel refuses these
        return None
    from automodel_amd.ops._backend import hip_ops

    ys = hip_ops().decode_rows(x.view(rows, K), ws, glu)
    return [y.view(*x.shape[:-1], y.shape[-1]) for y in ys]


def glu_rows(lins: list[nn.Module], x: torch.Tensor) -> torch.Tensor | None:
    """``silu(a) * b`` of the outputs a and b of two layers, or of the halves of one layer's, in one launch, for a prompt's
    many rows; None where that does not apply, and nothing is done."""
    if torch.compiler.is_compiling() or torch.is_grad_enabled():
        return None
    if not plain_linears(*lins) or any("forward" in lin.__dict__ for lin in lins):
        return None
    return gated(x, [lin.weight for lin in lins])


class DecodeLinear(nn.Linear):
    """nn.Linear that runs decode-shaped inputs on the in-tree GEMV."""

    @classmethod
    def from_linear(cls, lin: nn.Linear) -> "DecodeLinear":
        m = cls(lin.in_features, lin.out_features, bias=lin.bias is not None,
                device=lin.weight.device, dtype=lin.weight.dtype)
        with torch.no_grad():
            m.weight.copy_(lin.weight)
            if lin.bias is not None:
                m.bias.copy_(lin.bias)
        return m

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if _gemv_eligible(x, self.weight):
            lead = x.shape[:-1]
            y = gemv_bf16(x.reshape(-1, x.shape[-1]), self.weight, self.bias)
            return y.reshape(*lead, self.out_features)
        y = inferred(x, self.weight) if self.bias is None else None
        return F.linear(x, self.weight, self.bias) if y is None else y


def swap_linears_for_decode(model: nn.Module) -> int:
    """Swap every nn.Linear for DecodeLinear (weights shared by copy).
    Returns count. Call on an inference model before generate_graphed."""
    n = 0
    for name, parent in list(model.named_modules()):
        for child_name, child in list(parent.named_children()):
            if type(child) is nn.Linear:
                setattr(parent, child_name, DecodeLinear.from_linear(child))
                n += 1
    return n
