"""Context parallelism: zigzag sequence sharding + all-gather-KV attention.

Reference behavior: the reference ships five CP
mechanisms; the canonical MI355X one here is all-gather KV over the cp group
(RCCL all-gather over xGMI — for a single node the 7 direct links make one
large all-gather cheaper than per-step ring P2P) with zigzag (2-chunk
round-robin) load balancing exactly like ContextParallelSharder's "striped"
layout (context_parallel/sharder.py:116-143).

Each rank holds 2 chunks of S/(2P): chunk r and chunk 2P-1-r, so causal work
is balanced. Attention runs the in-tree flash kernel with ``q_start`` offsets
against the gathered KV; backward reduce-scatters dK/dV to their owners.
"""

from __future__ import annotations

from dataclasses import dataclass

import torch
import torch.distributed as dist

from automodel_amd.ops.attention import flash_attention


@dataclass
class CPContext:
    group: object
    rank: int
    world: int
    mechanism: str = "allgather"   # "allgather" (xGMI-preferred) | "ring"


_ACTIVE_CP: CPContext | None = None


def enable_cp(mesh_axis, mechanism: str = "allgather") -> CPContext:
    global _ACTIVE_CP
    assert mechanism in ("allgather", "ring"), mechanism
    group = mesh_axis.get_group() if hasattr(mesh_axis, "get_group") else mesh_axis
    _ACTIVE_CP = CPContext(group=group, rank=dist.get_rank(group),
                           world=dist.get_world_size(group),
                           mechanism=mechanism)
    return _ACTIVE_CP


def disable_cp() -> None:
    global _ACTIVE_CP
    _ACTIVE_CP = None


def active_cp() -> CPContext | None:
    return _ACTIVE_CP


def zigzag_chunk_ids(rank: int, world: int) -> tuple[int, int]:
    return rank, 2 * world - 1 - rank


def shard_batch_cp(batch: dict, rank: int, world: int, seq_dim: int = 1) -> dict:
    """Zigzag-shard input_ids/labels along seq; adds global position_ids."""
    if world == 1:
        return batch
    out = dict(batch)
    g0, g1 = zigzag_chunk_ids(rank, world)
    for key in ("input_ids", "labels", "attention_mask"):
        if key in batch and isinstance(batch[key], torch.Tensor):
            t = batch[key]
            S = t.shape[seq_dim]
            assert S % (2 * world) == 0, f"S={S} not divisible by 2*cp={2*world}"
            C = S // (2 * world)
            c0 = t.narrow(seq_dim, g0 * C, C)
            c1 = t.narrow(seq_dim, g1 * C, C)
            out[key] = torch.cat([c0, c1], dim=seq_dim)
    S = batch["input_ids"].shape[seq_dim]
    C = S // (2 * world)
    pos = torch.cat([
        torch.arange(g0 * C, (g0 + 1) * C),
        torch.arange(g1 * C, (g1 + 1) * C),
    ])
    B = batch["input_ids"].shape[0]
    out["position_ids"] = pos.unsqueeze(0).expand(B, -1).contiguous()
    return out


class _GatherSeqZigzag(torch.autograd.Function):
    """All-gather along seq and reorder zigzag chunks to global order.
    Backward: inverse reorder + reduce-scatter (sum) back to owners."""

    @staticmethod
    def forward(ctx, x: torch.Tensor, cp: CPContext):
        ctx.cp = cp
        P = cp.world
        B, S2, *rest = x.shape
        C = S2 // 2
        parts = [torch.empty_like(x) for _ in range(P)]
        dist.all_gather(parts, x.contiguous(), group=cp.group)
        stacked = torch.stack(parts)                      # [P, B, 2C, ...]
        chunks = stacked.view(P, B, 2, C, *rest)
        # global chunk g -> (rank, local slot)
        order = []
        for g in range(2 * P):
            r, slot = (g, 0) if g < P else (2 * P - 1 - g, 1)
            order.append(chunks[r, :, slot])
        return torch.cat(order, dim=1)                    # [B, 2P*C, ...]

    @staticmethod
    def backward(ctx, grad):
        cp = ctx.cp
        P = cp.world
        B, S, *rest = grad.shape
        C = S // (2 * P)
        g_chunks = grad.view(B, 2 * P, C, *rest)
        # rebuild per-rank zigzag layout [P, B, 2C, ...]
        per_rank = []
        for r in range(P):
            g0, g1 = zigzag_chunk_ids(r, P)
            per_rank.append(torch.cat([g_chunks[:, g0], g_chunks[:, g1]], dim=1))
        flat = torch.stack(per_rank).contiguous()         # [P, B, 2C, ...]
        if dist.get_backend(cp.group) == "gloo":
            dist.all_reduce(flat, group=cp.group)
            return flat[cp.rank], None
        out = torch.empty_like(flat[0])
        dist.reduce_scatter_tensor(out, flat, group=cp.group)
        return out, None


def cp_flash_attention(q, k, v, causal: bool = True, scale: float | None = None,
                       backend: str = "hip") -> torch.Tensor:
    """q/k/v local zigzag shards [B, 2C, H, D]; returns local O shard."""
    cp = _ACTIVE_CP
    assert cp is not None, "cp_flash_attention called without enable_cp"
    if cp.mechanism == "ring":
        return cp_ring_attention(q, k, v, causal=causal, scale=scale)
    P = cp.world
    B, S2 = q.shape[0], q.shape[1]
    C = S2 // 2
    kg = _GatherSeqZigzag.apply(k, cp)
    vg = _GatherSeqZigzag.apply(v, cp)
    g0, g1 = zigzag_chunk_ids(cp.rank, P)
    outs = []
    for local_slot, g in ((0, g0), (1, g1)):
        qc = q.narrow(1, local_slot * C, C)
        kv_len = (g + 1) * C if causal else 2 * P * C
        outs.append(
            flash_attention(qc, kg.narrow(1, 0, kv_len), vg.narrow(1, 0, kv_len),
                            causal=causal, scale=scale, backend=backend,
                            q_start=g * C)
        )
    return torch.cat(outs, dim=1)


def local_global_positions(rank: int, world: int, C: int,
                           device=None) -> torch.Tensor:
    """Global positions of this rank's 2C zigzag rows (chunk g0 then g1)."""
    g0, g1 = zigzag_chunk_ids(rank, world)
    return torch.cat([
        torch.arange(g0 * C, (g0 + 1) * C, device=device),
        torch.arange(g1 * C, (g1 + 1) * C, device=device),
    ])


def cp_blockdiag_attention(q, k, v, cu_seqlens: torch.Tensor,
                           scale: float | None = None) -> torch.Tensor:
    """Packed-document-correct CP attention (reference blockdiag_cp/
    exchange.py all-gather strategy + runtime.py cp_blockdiag_sdpa): each
    local (zigzag-sharded) q row attends only within its document AND
    causally, against the all-gathered global K/V. Doc boundaries come from
    the GLOBAL cu_seqlens, so they are exact regardless of how the shard
    cuts documents.

    GPU path: the native varlen flash kernel with per-token doc bounds and
    ``q_start`` — O(T) metadata, no dense mask, one launch per chunk.
    CPU path keeps the dense-mask sdpa reference (parity tests)."""
    import math

    cp = _ACTIVE_CP
    assert cp is not None, "cp_blockdiag_attention called without enable_cp"
    B, S2 = q.shape[0], q.shape[1]
    C = S2 // 2
    scale = scale if scale is not None else 1.0 / math.sqrt(q.shape[-1])
    kg = _GatherSeqZigzag.apply(k, cp)
    vg = _GatherSeqZigzag.apply(v, cp)
    T = kg.shape[1]
    dev = q.device

    if q.is_cuda and B == 1 and C % 128 == 0 and T % 32 == 0:
        from automodel_amd.ops.attention import _flash_hip, doc_bounds_from_cu

        ds, de = doc_bounds_from_cu(cu_seqlens.to(dev), T)
        g0, g1 = zigzag_chunk_ids(cp.rank, cp.world)
        outs = []
        for slot, g in ((0, g0), (1, g1)):
            qc = q.narrow(1, slot * C, C)
            outs.append(_flash_hip(qc, kg, vg, True, scale, g * C, ds, de, cu_seqlens.numel() - 1))
        return torch.cat(outs, dim=1)

    bounds = cu_seqlens.to(dev)[1:-1]
    doc_all = torch.bucketize(torch.arange(T, device=dev), bounds, right=True)
    gpos = local_global_positions(cp.rank, cp.world, C, device=dev)
    allowed = (doc_all[gpos][:, None] == doc_all[None, :]) \
        & (torch.arange(T, device=dev)[None, :] <= gpos[:, None])
    mask = torch.where(allowed, 0.0, float("-inf")) \
        .to(q.dtype).reshape(1, 1, S2, T)

    from automodel_amd.ops.attention import sdpa_masked

    return sdpa_masked(q, kg, vg, mask, scale)


# ===========================================================================
# Ring-P2P KV context parallelism (reference's ring exchange strategy,
# context_parallel/exchange.py ring mode). Peak KV memory is O(S/P) per step instead of the all-gather
# path's O(S): each rank's zigzag KV block rotates around the cp ring
# (P2P isend/irecv — on xGMI these ride the direct per-pair links), and
# attention partials merge by online softmax in fp32. Backward makes the
# same P-step rotation, accumulating dq locally while dK/dV accumulators
# travel WITH their KV block and hop home on a final rotation. Exact (same
# math as flash): parity-tested against cp_flash_attention on gloo world 2.
# ===========================================================================


def _ring_sendrecv(bufs: list[torch.Tensor], cp: CPContext) -> list[torch.Tensor]:
    """Rotate tensors one hop: send to rank+1, receive from rank-1."""
    dst = (cp.rank + 1) % cp.world
    src = (cp.rank - 1) % cp.world
    outs = [torch.empty_like(b) for b in bufs]
    reqs = []
    for b, o in zip(bufs, outs):
        reqs.append(dist.P2POp(dist.isend, b.contiguous(), dst, group=cp.group))
        reqs.append(dist.P2POp(dist.irecv, o, src, group=cp.group))
    for w in dist.batch_isend_irecv(reqs):
        w.wait()
    return outs


def _ring_pairs(qg: tuple[int, int], kg: tuple[int, int], causal: bool):
    for qi in (0, 1):
        for ki in (0, 1):
            if causal and kg[ki] > qg[qi]:
                continue
            yield qi, ki, causal and kg[ki] == qg[qi]


class _RingAttention(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, cp, causal, scale):
        P, r = cp.world, cp.rank
        B, S2, H, D = q.shape
        C = S2 // 2
        qg = zigzag_chunk_ids(r, P)
        qf = q.float().view(B, 2, C, H, D)
        m = torch.full((B, 2, C, H), float("-inf"), device=q.device)
        den = torch.zeros_like(m)
        num = torch.zeros(B, 2, C, H, D, device=q.device)
        Hk = k.shape[2]
        rep = H // Hk
        kb, vb = k.float().view(B, 2, C, Hk, D), v.float().view(B, 2, C, Hk, D)
        diag = torch.ones(C, C, dtype=torch.bool, device=q.device).triu(1)
        for step in range(P):
            src = (r - step) % P
            kg = zigzag_chunk_ids(src, P)
            for qi, ki, is_diag in _ring_pairs(qg, kg, causal):
                ke = kb[:, ki].repeat_interleave(rep, dim=2) if rep > 1 else kb[:, ki]
                ve = vb[:, ki].repeat_interleave(rep, dim=2) if rep > 1 else vb[:, ki]
                s = torch.einsum("bqhd,bkhd->bqkh", qf[:, qi], ke) * scale
                if is_diag:
                    s = s.masked_fill(diag.view(1, C, C, 1), float("-inf"))
                bm = s.amax(dim=2)
                newm = torch.maximum(m[:, qi], bm)
                p = torch.exp(s - newm.unsqueeze(2))
                corr = torch.exp(m[:, qi] - newm)
                den[:, qi] = den[:, qi] * corr + p.sum(dim=2)
                num[:, qi] = (num[:, qi] * corr.unsqueeze(-1)
                              + torch.einsum("bqkh,bkhd->bqhd", p, ve))
                m[:, qi] = newm
            if step < P - 1:
                kb, vb = _ring_sendrecv([kb, vb], cp)
        o = num / den.clamp_min(1e-30).unsqueeze(-1)
        lse = m + den.clamp_min(1e-30).log()
        ctx.save_for_backward(q, k, v, o.to(q.dtype), lse)
        ctx.cp, ctx.causal, ctx.scale = cp, causal, scale
        return o.view(B, S2, H, D).to(q.dtype)

    @staticmethod
    def backward(ctx, do):
        q, k, v, o, lse = ctx.saved_tensors
        cp, causal, scale = ctx.cp, ctx.causal, ctx.scale
        P, r = cp.world, cp.rank
        B, S2, H, D = q.shape
        C = S2 // 2
        qg = zigzag_chunk_ids(r, P)
        qf = q.float().view(B, 2, C, H, D)
        dof = do.float().view(B, 2, C, H, D)
        of = o.float().view(B, 2, C, H, D)
        Dm = (dof * of).sum(-1)                    # [B, 2, C, H]
        dq = torch.zeros_like(qf)
        Hk = k.shape[2]
        rep = H // Hk
        kb, vb = k.float().view(B, 2, C, Hk, D), v.float().view(B, 2, C, Hk, D)
        dkb, dvb = torch.zeros_like(kb), torch.zeros_like(vb)
        diag = torch.ones(C, C, dtype=torch.bool, device=q.device).triu(1)

        def fold(t):   # [B, C, H, D] -> [B, C, Hk, D] (sum over GQA reps)
            return t if rep == 1 else t.view(B, C, Hk, rep, D).sum(3)

        for step in range(P):
            src = (r - step) % P
            kg = zigzag_chunk_ids(src, P)
            for qi, ki, is_diag in _ring_pairs(qg, kg, causal):
                ke = kb[:, ki].repeat_interleave(rep, dim=2) if rep > 1 else kb[:, ki]
                ve = vb[:, ki].repeat_interleave(rep, dim=2) if rep > 1 else vb[:, ki]
                s = torch.einsum("bqhd,bkhd->bqkh", qf[:, qi], ke) * scale
                if is_diag:
                    s = s.masked_fill(diag.view(1, C, C, 1), float("-inf"))
                p = torch.exp(s - lse[:, qi].unsqueeze(2))
                dvb[:, ki] += fold(torch.einsum("bqkh,bqhd->bkhd", p, dof[:, qi]))
                dp = torch.einsum("bqhd,bkhd->bqkh", dof[:, qi], ve)
                ds = p * (dp - Dm[:, qi].unsqueeze(2)) * scale
                dq[:, qi] += torch.einsum("bqkh,bkhd->bqhd", ds, ke)
                dkb[:, ki] += fold(torch.einsum("bqkh,bqhd->bkhd", ds, qf[:, qi]))
            # rotate kv + their grad accumulators together; the final hop
            # returns each block's dK/dV to its owner
            kb, vb, dkb, dvb = _ring_sendrecv([kb, vb, dkb, dvb], cp)
        return (dq.view(B, S2, H, D).to(q.dtype),
                dkb.view(B, S2, Hk, D).to(k.dtype),
                dvb.view(B, S2, Hk, D).to(v.dtype), None, None, None)


def cp_ring_attention(q, k, v, causal: bool = True,
                      scale: float | None = None) -> torch.Tensor:
    """Ring-P2P CP attention over zigzag shards [B, 2C, H, D] -> local O.
    Memory-bounded alternative to cp_flash_attention (KV never gathered)."""
    import math

    cp = _ACTIVE_CP
    assert cp is not None, "cp_ring_attention called without enable_cp"
    scale = scale if scale is not None else 1.0 / math.sqrt(q.shape[-1])
    if cp.world == 1:
        return flash_attention(q, k, v, causal=causal, scale=scale,
                               backend="torch")
    return _RingAttention.apply(q, k, v, cp, causal, scale)
