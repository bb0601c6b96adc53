"""Latent attention as a module, for packed tokens, with or without a cache."""

from __future__ import annotations

import torch
import torch.nn as nn

from automodel_amd.ops.latent_attention import (
    MFMA_MAX_CACHE_WIDTH,
    MFMA_MAX_RANK,
    LatentAttentionSpec,
    PackedStep,
    decode_splits,
    latent_attention_decode,
    latent_attention_prompt,
)
from automodel_amd.ops.residual_norm import use_hip
from automodel_amd.ops.rms_norm import RMSNorm
from automodel_amd.serving.decode_linear import plain_linears, project, unobserved


class LatentAttention(nn.Module):
    """h [T, width] -> [T, width].

    ``q_kv_a_proj`` stacks the query projection and the latent/rotated-key
    down-projection (one GEMM per layer); ``kv_b_proj`` stacks the key and the
    value up-projection.
    """

    def __init__(self, width: int, spec: LatentAttentionSpec, norm_backend: str = "hip"):
        super().__init__()
        self.spec = spec
        self.q_kv_a_proj = nn.Linear(width, spec.q_width + spec.kv_rank + spec.rot_dim, bias=False)
        self.kv_a_layernorm = RMSNorm(spec.kv_rank, spec.eps, norm_backend)
        self.kv_b_proj = nn.Linear(spec.kv_rank, spec.heads * (spec.dim + spec.vdim), bias=False)
        self.o_proj = nn.Linear(spec.heads * spec.vdim, width, bias=False)

    def forward(self, h: torch.Tensor, step: PackedStep, rope: tuple[torch.Tensor, torch.Tensor],
                cache: torch.Tensor | None = None) -> torch.Tensor:
        if type(self.kv_b_proj) is not nn.Linear and cache is not None:
            # the cached path multiplies by the raw weight (absorbed form)
            raise RuntimeError("merge adapters on kv_b_proj before decoding with a cache")
        qkv = project(self.q_kv_a_proj, h)
        attend = latent_attention_prompt if step.prompt else latent_attention_decode
        o = attend(qkv, self.kv_a_layernorm.weight, self.kv_b_proj.weight, self.spec, rope,
                   step, cache)
        return project(self.o_proj, o)

    def decode_layer(self, layer: nn.Module, x: torch.Tensor, h: torch.Tensor,
                     next_norm: torch.Tensor | None, step: PackedStep,
                     rope: tuple[torch.Tensor, torch.Tensor], cache: torch.Tensor | None = None
                     ) -> tuple[torch.Tensor, torch.Tensor | None] | None:
        """``layer``'s whole forward for a decode step, all kernels issued by one native call
        (csrc/latent_layer.cpp); None where that does not apply, and nothing is done."""
        from automodel_amd.models.common.blocks import SquaredReluMLP

        spec, mlp = self.spec, layer.mlp
        if not (cache is not None and not step.prompt and use_hip(h)
                and h.dtype == torch.bfloat16 and type(h) is type(x) is torch.Tensor
                and spec.kv_rank <= MFMA_MAX_RANK and spec.cache_width <= MFMA_MAX_CACHE_WIDTH
                and type(self) is LatentAttention and type(mlp) in (type(None), SquaredReluMLP)
                and unobserved(self, *([] if mlp is None else [mlp]))):
            return None
        lins = [self.q_kv_a_proj, self.kv_b_proj, self.o_proj]
        if not plain_linears(*lins, *([] if mlp is None else [mlp.up_proj, mlp.down_proj])):
            return None
        ws = [lins[0].weight, self.kv_a_layernorm.weight, lins[1].weight, lins[2].weight,
              layer.post_attention_layernorm.weight]
        if mlp is not None:
            ws += [layer.pre_feedforward_layernorm.weight, mlp.up_proj.weight,
                   mlp.down_proj.weight, layer.post_feedforward_layernorm.weight]
        from automodel_amd.ops._backend import hip_ops

        out = hip_ops().latent_decode_layer(
            x, h, ws, next_norm, rope[0], rope[1], step.positions, step.slots, cache, layer.eps,
            spec.eps, layer.mult, spec.scale, spec.heads, spec.dim, spec.rot_dim,
            decode_splits(h.shape[0], spec.heads, cache.shape[1]))
        if not out:
            return None
        return x, (out[0] if next_norm is not None else None)
