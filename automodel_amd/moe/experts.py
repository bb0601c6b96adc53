"""Grouped expert compute: stacked weights, token permute, grouped GEMM.

Reference behavior: nemo_automodel/components/moe/experts.py:370-876
(GroupedExperts with loop / torch._grouped_mm paths; GroupedExpertsDeepEP
permute -> grouped GEMM -> activation -> grouped GEMM -> unpermute).

Weights are stacked [E, ...] tensors so EP sharding is a dim-0 DTensor shard
and HF per-expert keys map via the model's state_dict_adapter.
"""

from __future__ import annotations

import torch
import torch.nn as nn

from automodel_amd.ops._backend import followed
from automodel_amd.ops.linear import _ordinary
from automodel_amd.ops.swiglu import swiglu


def permute_tokens(x: torch.Tensor, indices: torch.Tensor, n_experts: int):
    """Sort token replicas by expert. Returns (x_perm [T*K, H], sort_idx,
    tokens_per_expert [E])."""
    T, K = indices.shape
    flat = indices.reshape(-1)
    sort_idx = flat.argsort(stable=True)
    counts = torch.bincount(flat, minlength=n_experts)
    x_rep = x.repeat_interleave(K, dim=0)
    return x_rep[sort_idx], sort_idx, counts


class _FusedPermuteGather(torch.autograd.Function):
    """x [T,H] -> x_perm [T*K,H] via the HIP kernel that writes each token's copies (no
    repeat_interleave copy). Backward: per-token sum of replica grads via
    the combine kernel without probs."""

    @staticmethod
    def forward(ctx, x, pos, K):
        from automodel_amd.ops._backend import hip_ops

        ctx.save_for_backward(pos)
        ctx.K = K
        return hip_ops().permute_rows(x.contiguous(), pos.view(-1, K))

    @staticmethod
    def backward(ctx, g):
        from automodel_amd.ops._backend import hip_ops

        (pos,) = ctx.saved_tensors
        dx = hip_ops().unpermute_sum(g.contiguous(), pos.view(-1, ctx.K))
        return dx, None, None


_ROUTE_MAX_EXPERTS = 4096       # csrc/moe_kernels.hip


def check_experts(indices: torch.Tensor, n_experts: int) -> None:
    """Refuses experts that do not exist; waits for the device that ``indices`` is on."""
    if indices.numel():
        low, high = torch.stack(indices.aminmax()).tolist()
        if low < 0 or high >= n_experts:
            raise RuntimeError(f"experts {low} to {high} chosen of {n_experts}")


def _route(x, probs, indices, n_experts, checked):
    """(counts, order, src, pos, perm_probs, probs32): where each choice's row is, on the device. Nothing
    waits for the host where ``checked`` says that every index is one of an expert; without it the indices
    are looked at first."""
    from automodel_amd.ops._backend import hip_ops

    if not checked:
        check_experts(indices, n_experts)
    T, K = indices.shape
    with torch.no_grad():
        probs32 = probs.detach().float().contiguous()
        if n_experts <= _ROUTE_MAX_EXPERTS:
            counts, order, src, pos, perm_probs = hip_ops().route_plan(
                indices.long().contiguous(), probs32, n_experts)
        else:
            order = indices.reshape(-1).argsort(stable=True)
            counts = torch.bincount(indices.reshape(-1), minlength=n_experts).to(torch.int32)
            src = (order // K).to(torch.int32)
            pos = torch.empty_like(order)
            pos[order] = torch.arange(T * K, device=x.device)
            pos, order = pos.to(torch.int32).view(T, K), order.to(torch.int32)
            perm_probs = probs32.reshape(-1)[order]
    return counts, order, src, pos, perm_probs, probs32


def fused_dispatch_combine(x, probs, indices, n_experts, expert_fn, checked=False):
    """GPU MoE glue: device-side routing plan, HIP gather, expert_fn over permuted
    rows, HIP combine — one gather + one combine instead of
    repeat_interleave + fancy-index + scatter (reference fused permute/
    unpermute, moe_utils.py:31/115)."""
    counts, order, src, pos, perm_probs, probs32 = _route(x, probs, indices, n_experts, checked)
    x_perm = _FusedPermuteGather.apply(x, pos, indices.shape[1])
    y_perm = expert_fn(x_perm, counts)
    return _CombineWithProbs.apply(y_perm, pos, probs, src, perm_probs, order, probs32)


class _Experts(torch.autograd.Function):
    """Gated experts from the tokens to their weighted sum, as one function: a step of 1000 tokens and few experts, which
    waits for the host, takes 0.88 of the time of one function each for copies, products, activation and sum.

    Where ``inner``, the backward does without the experts' outputs. With dh the gradient of an unweighted row's activation
    h, a choice's weight has the gradient dh h, a sum over the inner width, and the weighted row p h is the operand of
    the last weight's gradient (csrc/swiglu.hip). That moves two rows of the hidden width less and one of the inner
    width more: with hidden widths of twice the inner and more 0.96 to 1.06 of the time of forward and backward, 0.99 in the
    mean, below 0.94 to 1.04 and 1.00 (826 layers of 500 to 8200 tokens, 8 to 128 experts:
    profiles/sweep_experts_backward.csv)."""

    @staticmethod
    def forward(ctx, x, probs, gate, up, down, order, src, pos, perm_probs, probs32, offs, tile_map, n_tiles, bm):
        from automodel_amd.ops._backend import hip_ops

        ops, plan = hip_ops(), (offs, tile_map, n_tiles, bm)
        gate, up, down = gate.contiguous(), up.contiguous(), down.contiguous()
        rows = ops.permute_rows(x.contiguous(), pos)
        g, u, h = ops.grouped_glu(rows, gate, up, *plan)
        y = ops.grouped_gemm_nt(h, down, *plan)
        ctx.inner = x.shape[1] >= 2 * gate.shape[1]
        ctx.save_for_backward(rows, g, u, gate, up, down, order, src, pos, perm_probs, offs, tile_map, n_tiles,
                              *(() if ctx.inner else (h, y)))
        ctx.bm, ctx.probs = bm, (probs.shape, probs.dtype)
        return ops.unpermute_combine(y, pos, probs32)

    @staticmethod
    def backward(ctx, d):
        from automodel_amd.ops._backend import hip_ops

        rows, g, u, gate, up, down, order, src, pos, perm_probs, offs, tile_map, n_tiles, *kept = ctx.saved_tensors
        ops, plan, need = hip_ops(), (offs, tile_map, n_tiles, ctx.bm), ctx.needs_input_grad
        E = gate.shape[0]
        if ctx.inner:
            d = ops.permute_rows(d.contiguous(), pos)
            dg, du, h, dp = ops.swiglu_rows_bwd(ops.grouped_gemm_nn(d, down, *plan), g, u, perm_probs, order)
        else:
            h, y = kept
            d, dp = ops.combine_bwd(d.contiguous(), y, src, order, perm_probs)
            dh = ops.grouped_gemm_nn(d, down, *plan)
        d_down = ops.grouped_gemm_tn(d, h, offs, E) if need[4] else None
        del d, h
        if not ctx.inner:
            dg, du = ops.swiglu_bwd(dh, g, u)
        dx = ops.grouped_gemm_nn2(dg, gate, du, up, *plan) if need[0] else None
        d_gate = ops.grouped_gemm_tn(dg, rows, offs, E) if need[2] else None
        d_up = ops.grouped_gemm_tn(du, rows, offs, E) if need[3] else None
        if need[0]:
            dx = ops.unpermute_sum(dx, pos)
        shape, dtype = ctx.probs
        return dx, dp.view(shape).to(dtype) if need[1] else None, d_gate, d_up, d_down, *[None] * 9


class _CombineWithProbs(torch.autograd.Function):
    @staticmethod
    def forward(ctx, y_perm, pos, probs, src, perm_probs, order, probs32):
        from automodel_amd.ops._backend import hip_ops

        y_perm = y_perm.contiguous()
        out = hip_ops().unpermute_combine(y_perm, pos, probs32)
        ctx.save_for_backward(y_perm, src, perm_probs, order)
        ctx.probs_shape, ctx.probs_dtype = probs.shape, probs.dtype
        return out

    @staticmethod
    def backward(ctx, g):
        from automodel_amd.ops._backend import hip_ops

        y_perm, src, perm_probs, order = ctx.saved_tensors
        dy, dprobs = hip_ops().combine_bwd(g.contiguous(), y_perm, src, order, perm_probs)
        return dy, None, dprobs.view(ctx.probs_shape).to(ctx.probs_dtype), None, None, None, None


def unpermute_tokens(y_perm: torch.Tensor, sort_idx: torch.Tensor,
                     probs: torch.Tensor) -> torch.Tensor:
    """Scatter back and combine top-k with routing probs."""
    T, K = probs.shape
    y = torch.empty_like(y_perm)
    y[sort_idx] = y_perm
    y = y.view(T, K, -1)
    return (y * probs.unsqueeze(-1)).sum(dim=1)


class GroupedExperts(nn.Module):
    def __init__(self, n_experts: int, hidden_size: int, intermediate_size: int,
                 backend: str = "auto"):
        super().__init__()
        self.n_experts = n_experts
        self.hidden_size = hidden_size
        self.intermediate_size = intermediate_size
        self.backend = backend
        self.gate_proj = nn.Parameter(torch.empty(n_experts, intermediate_size, hidden_size))
        self.up_proj = nn.Parameter(torch.empty(n_experts, intermediate_size, hidden_size))
        self.down_proj = nn.Parameter(torch.empty(n_experts, hidden_size, intermediate_size))
        # opt-in fp8 expert forward (set by quantization.fp8.apply_fp8 /
        # bench --fp8): fp8-e4m3 grouped NT forward with delayed tensorwise
        # scaling, bf16 grouped backward
        self.fp8 = False
        self._fp8_states = None

    def init_weights(self, std: float = 0.02) -> None:
        for p in (self.gate_proj, self.up_proj, self.down_proj):
            nn.init.normal_(p, std=std)

    @staticmethod
    def project(x_perm: torch.Tensor, w: torch.Tensor, counts) -> torch.Tensor:
        """Grouped projection y[t] = x[t] @ w[expert(t)].T over expert-sorted
        tokens — grouped-GEMM HIP kernel on GPU, per-expert loop on CPU.
        (Also used by peft/lora_experts.py adapters.)"""
        if (x_perm.is_cuda and x_perm.dtype == torch.bfloat16
                and x_perm.numel() > 0):
            from automodel_amd.ops.grouped_gemm import grouped_linear

            return grouped_linear(x_perm, w, counts)
        cl = counts.tolist() if torch.is_tensor(counts) else list(counts)
        outs = []
        start = 0
        for e, n in enumerate(cl):
            if n == 0:
                continue
            outs.append(x_perm[start : start + n] @ w[e].t())
            start += n
        return torch.cat(outs, dim=0) if outs else x_perm[:0]

    def _expert_mlp_loop(self, x_perm: torch.Tensor, counts: torch.Tensor) -> torch.Tensor:
        outs = []
        start = 0
        counts_list = counts.tolist()
        for e, n in enumerate(counts_list):
            if n == 0:
                continue
            xe = x_perm[start : start + n]
            h = swiglu(xe @ self.gate_proj[e].t(), xe @ self.up_proj[e].t())
            outs.append(h @ self.down_proj[e].t())
            start += n
        return torch.cat(outs, dim=0) if outs else x_perm[:0]

    def forward_permuted(self, x_perm: torch.Tensor, counts: torch.Tensor) -> torch.Tensor:
        """Compute experts over tokens already sorted by expert (counts[e] each).

        counts covers THIS module's experts (post-EP-shard slice). On GPU the
        three projections run the in-tree grouped-GEMM HIP kernel.
        """
        use_grouped = (
            x_perm.is_cuda and self.backend in ("auto", "hip_grouped")
            and x_perm.dtype == torch.bfloat16
            and self.intermediate_size % 128 == 0 and self.hidden_size % 128 == 0
            and x_perm.numel() > 0
        )
        if use_grouped:
            from automodel_amd.ops.grouped_gemm import (
                grouped_linear,
                grouped_linear_pair,
                make_group_plan,
                tile_rows,
            )

            if torch.is_tensor(counts) and counts.is_cuda:
                # device-side plan shared by all three projections — the
                # routing counts never touch the host; the fp8 kernels have
                # 256-row tiles when every projection width allows
                if self.fp8:
                    bm = 256 if (self.intermediate_size % 256 == 0
                                 and self.hidden_size % 256 == 0) else 128
                else:
                    bm = tile_rows(x_perm.shape[0], self.n_experts, self.intermediate_size,
                                   self.hidden_size)
                plan = (*make_group_plan(counts, x_perm.shape[0], bm), bm)
                cl = counts
            else:
                plan = None
                cl = counts.tolist() if torch.is_tensor(counts) else list(counts)
            if (self.fp8 and plan is not None
                    and self.intermediate_size % 128 == 0
                    and self.hidden_size % 128 == 0):
                from automodel_amd.ops.grouped_gemm import (
                    Fp8GroupedState,
                    grouped_linear_fp8,
                )

                if self._fp8_states is None:
                    self._fp8_states = {k: Fp8GroupedState()
                                        for k in ("gate", "up", "down")}
                st = self._fp8_states
                from automodel_amd.ops._backend import hip_ops

                xc = x_perm.contiguous()
                # non-differentiable byproducts: cast under no_grad so the
                # fp8 bytes don't drag an autograd-fallback node into BOTH
                # gate and up Function graphs
                with torch.no_grad():
                    sx = st["gate"].x_scale(xc)
                    x8 = hip_ops().fp8_cast(xc, sx, st["gate"].amax_x, False)
                g = grouped_linear_fp8(xc, self.gate_proj, cl, plan,
                                       st["gate"], x8, sx)
                u = grouped_linear_fp8(xc, self.up_proj, cl, plan,
                                       st["up"], x8, sx)
                h = swiglu(g, u)
                return grouped_linear_fp8(h, self.down_proj, cl, plan, st["down"])
            if plan is not None:
                g, u = grouped_linear_pair(x_perm, self.gate_proj, self.up_proj, cl, plan)
            else:
                g = grouped_linear(x_perm, self.gate_proj, cl)
                u = grouped_linear(x_perm, self.up_proj, cl)
            h = swiglu(g, u)
            return grouped_linear(h, self.down_proj, cl, plan=plan)
        return self._expert_mlp_loop(x_perm, counts)

    def _as_one(self, x: torch.Tensor, probs: torch.Tensor) -> bool:
        """Whether the layer can be one function: plain bf16 experts that the kernels take, and nothing
        that has a part of them replaced or follows the operations."""
        ws = (self.gate_proj, self.up_proj, self.down_proj)
        return (not followed() and type(self).forward_permuted is GroupedExperts.forward_permuted
                and "forward_permuted" not in self.__dict__ and not self.fp8
                and self.intermediate_size % 128 == 0 and self.hidden_size % 128 == 0
                and x.dim() == 2 and x.numel() > 0 and probs.numel() > 0 and probs.is_floating_point()
                and all(type(w) in (torch.Tensor, nn.Parameter) and w.dtype == x.dtype and w.device == x.device for w in ws)
                and ws[0].shape == ws[1].shape == (self.n_experts, self.intermediate_size, self.hidden_size)
                and ws[2].shape == (self.n_experts, self.hidden_size, self.intermediate_size)
                and x.shape[1] == self.hidden_size and _ordinary(x, probs))

    def forward(self, x: torch.Tensor, probs: torch.Tensor, indices: torch.Tensor,
                checked: bool = False) -> torch.Tensor:
        """``checked``: the caller knows that every index is one of an expert."""
        if (x.is_cuda and x.dtype == torch.bfloat16 and x.shape[-1] % 8 == 0
                and self.backend in ("auto", "hip_grouped")):
            if self._as_one(x, probs):
                from automodel_amd.ops.grouped_gemm import make_group_plan, tile_rows

                counts, order, src, pos, perm_probs, probs32 = _route(x, probs, indices, self.n_experts, checked)
                M = indices.numel()
                bm = tile_rows(M, self.n_experts, self.intermediate_size, self.hidden_size)
                return _Experts.apply(x, probs, self.gate_proj, self.up_proj, self.down_proj, order, src, pos,
                                      perm_probs, probs32, *make_group_plan(counts, M, bm), bm)
            return fused_dispatch_combine(x, probs, indices, self.n_experts,
                                          self.forward_permuted, checked)
        x_perm, sort_idx, counts = permute_tokens(x, indices, self.n_experts)
        y_perm = self.forward_permuted(x_perm, counts)
        return unpermute_tokens(y_perm, sort_idx, probs)
