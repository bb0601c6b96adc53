"""Decoder building blocks around a 32-bit residual stream.

* ``SquaredReluMLP``: up -> max(x, 0)^2 -> down.
* ``ClampedGluMLP``: [gate; up] -> clamped gated unit -> down.
* ``HyperConnection``: a sublayer's input norm and its weights towards several
  residual streams (``ops/hyper.py``).
* ``SandwichLayer``: every sublayer is normed before and after, and enters the
  residual with a constant factor. Consecutive layers hand the next normed
  input along, so that each residual update is one fused kernel.
* ``layer_schedule`` / ``LoopInput``: a stretch of layers run several times with
  shared weights, each pass starting from a projection of the current stream
  and the embedding output.
"""

from __future__ import annotations

import torch
import torch.nn as nn

from automodel_amd.ops.hyper import clamped_glu, hyper_step
from automodel_amd.ops.residual_norm import concat_cast, residual_add_norm
from automodel_amd.ops.rms_norm import RMSNorm
from automodel_amd.serving.decode_linear import project


class SquaredReluMLP(nn.Module):
    def __init__(self, width: int, inter: int):
        super().__init__()
        self.up_proj = nn.Linear(width, inter, bias=False)
        self.down_proj = nn.Linear(inter, width, bias=False)

    def forward(self, h: torch.Tensor) -> torch.Tensor:
        return project(self.down_proj, project(self.up_proj, h, relu2=True))


class ClampedGluMLP(nn.Module):
    """``gate_up_proj`` stacks the gate and the up projection."""

    def __init__(self, width: int, inter: int, limit: float, alpha: float = 1.702):
        super().__init__()
        self.limit, self.alpha = limit, alpha
        self.gate_up_proj = nn.Linear(width, 2 * inter, bias=False)
        self.down_proj = nn.Linear(inter, width, bias=False)

    def forward(self, h: torch.Tensor) -> torch.Tensor:
        return project(self.down_proj, clamped_glu(project(self.gate_up_proj, h), self.limit,
                                                   self.alpha))


class HyperConnection(nn.Module):
    """Around one sublayer: ``norm`` and ``w_in`` [streams] make its input,
    ``w_mix`` [from, to] and ``w_out`` [streams] the streams after it."""

    def __init__(self, width: int, streams: int, eps: float, norm_backend: str = "hip"):
        super().__init__()
        self.eps = eps
        self.norm = RMSNorm(width, eps, norm_backend)
        self.w_in = nn.Parameter(torch.full((streams,), 1.0 / streams))
        self.w_out = nn.Parameter(torch.ones(streams))
        self.w_mix = nn.Parameter(torch.eye(streams))

    def update(self, x, y, nxt: "HyperConnection | None", final_norm, keep: bool = True):
        """Streams after this sublayer's output y, and the input of the next one
        (or, without, the normed sum of the streams)."""
        w_in, w_norm = (None, final_norm) if nxt is None else (nxt.w_in, nxt.norm.weight)
        return hyper_step(x, y, self.w_mix, self.w_out, w_in, w_norm, self.eps, keep)


class SandwichLayer(nn.Module):
    """x += mult * post(sublayer(pre(x))) for the mixer and, if there is one,
    the feed-forward.

    ``forward(x, h, next_norm, *mixer_args)``: x is the float32 residual, h its
    normed form for the mixer, ``next_norm`` the norm that the following layer
    applies first (None if something else comes in between). Returns the new
    ``(x, h)``, h being None when there is no ``next_norm``.
    """

    def __init__(self, width: int, mixer: nn.Module, mlp: nn.Module | None, eps: float,
                 mult: float = 1.0, norm_backend: str = "hip"):
        super().__init__()
        self.eps, self.mult = eps, mult
        self.input_layernorm = RMSNorm(width, eps, norm_backend)
        self.self_attn = mixer
        self.post_attention_layernorm = RMSNorm(width, eps, norm_backend)
        self.mlp = mlp
        if mlp is not None:
            self.pre_feedforward_layernorm = RMSNorm(width, eps, norm_backend)
            self.post_feedforward_layernorm = RMSNorm(width, eps, norm_backend)

    def forward(self, x: torch.Tensor, h: torch.Tensor, next_norm: torch.Tensor | None,
                *mixer_args) -> tuple[torch.Tensor, torch.Tensor | None]:
        decode = getattr(self.self_attn, "decode_layer", None)
        done = decode(self, x, h, next_norm, *mixer_args) if decode is not None else None
        if done is not None:
            return done
        y = self.self_attn(h, *mixer_args)
        if self.mlp is None:
            return residual_add_norm(x, y, self.post_attention_layernorm.weight, self.mult,
                                     self.eps, next_norm)
        x, h = residual_add_norm(x, y, self.post_attention_layernorm.weight, self.mult,
                                 self.eps, self.pre_feedforward_layernorm.weight)
        return residual_add_norm(x, self.mlp(h), self.post_feedforward_layernorm.weight,
                                 self.mult, self.eps, next_norm)


def layer_schedule(n_layers: int, loop: dict | None = None) -> list[tuple[int, bool]]:
    """Execution order as (layer index, a pass of the loop begins here).

    ``loop`` = {start, stop, times}: layers start..stop-1 run ``times`` times
    in a row before the rest follow.
    """
    if not loop:
        return [(i, False) for i in range(n_layers)]
    start, stop, times = int(loop["start"]), int(loop["stop"]), int(loop["times"])
    if not (0 <= start < stop <= n_layers and times >= 1):
        raise ValueError(f"loop {loop} does not fit {n_layers} layers")
    one_pass = [(i, i == start) for i in range(start, stop)]
    return ([(i, False) for i in range(start)] + one_pass * times
            + [(i, False) for i in range(stop, n_layers)])


class LoopInput(nn.Module):
    """x <- W [x ; x0], in and out in float32."""

    def __init__(self, width: int):
        super().__init__()
        self.proj = nn.Linear(2 * width, width, bias=False)

    def forward(self, x: torch.Tensor, x0: torch.Tensor) -> torch.Tensor:
        return project(self.proj, concat_cast(x, x0, self.proj.weight.dtype), out_f32=True)
