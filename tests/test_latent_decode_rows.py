"""Decode-side latent attention: both projections over row groups, ragged ranks and head dims."""

import pytest
import torch

from automodel_amd.ops.latent_attention import pad32

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def bf16_close(got, want):
    # rounded once to 8 bits; float32 sums add far less than 1e-5 of the largest
    err = (got.double() - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 1e-5 * want.abs().max()).all(), float(err.max())


@pytest.mark.parametrize("R", [1, 2, 5, 16, 17, 33])
@pytest.mark.parametrize("H,dn,dr,rank", [
    (3, 32, 8, 64), (2, 128, 64, 512), (5, 160, 16, 72), (1, 256, 32, 200), (2, 48, 16, 64),
    (2, 64, 6, 40),
])
def test_prep(R, H, dn, dr, rank):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    n_slots, max_len = R + 2, 9
    qkv = torch.randn(R, H * (dn + dr) + rank + dr, device="cuda").bfloat16()
    w = (torch.randn(H * dn, rank, device="cuda") * dn ** -0.5).bfloat16()
    norm = (1 + 0.1 * torch.randn(rank, device="cuda")).bfloat16()
    angle = torch.randn(max_len, dr // 2, device="cuda")
    cos, sin = angle.cos(), angle.sin()
    pos = torch.randint(0, max_len, (R,), device="cuda", dtype=torch.int32)
    slot = torch.randperm(n_slots, device="cuda")[:R].int()
    slot[R // 2] = -1 if R > 1 else 0                   # not written
    RP, C = pad32(rank), pad32(rank) + pad32(dr)
    cache = torch.full((n_slots, max_len, C), 7.0, device="cuda").bfloat16()
    before = cache.clone()
    q = hip_ops().latent_decode_prep(qkv, w, norm, 1e-6, cos, sin, pos, slot, cache, H, dn, dr)

    def turn(x, p):
        c, s = cos[p.long()].double(), sin[p.long()].double()
        while c.dim() < x.dim():
            c, s = c[:, None], s[:, None]
        a, b = x.double().split(dr // 2, -1)
        return torch.cat([a * c - b * s, b * c + a * s], -1)

    heads = qkv[:, :H * (dn + dr)].view(R, H, dn + dr)
    want = torch.zeros(R, H, C, device="cuda", dtype=torch.float64)
    for h in range(H):
        want[:, h, :rank] = heads[:, h, :dn].double() @ w[h * dn:(h + 1) * dn].double()
    want[:, :, RP:RP + dr] = turn(heads[:, :, dn:], pos)
    bf16_close(q, want)
    x = qkv[:, H * (dn + dr):].double()
    c = x[:, :rank] * torch.rsqrt((x[:, :rank] ** 2).mean(-1, keepdim=True) + 1e-6) * norm.double()
    for r in range(R):
        if slot[r] >= 0:
            row = cache[slot[r], pos[r]]
            bf16_close(row[:rank], c[r])
            bf16_close(row[RP:RP + dr], turn(x[r:r + 1, rank:], pos[r:r + 1])[0])
            before[slot[r], pos[r]] = row
    assert torch.equal(cache, before)


@pytest.mark.parametrize("R,S", [(1, 1), (1, 4), (1, 24), (2, 10), (5, 3), (7, 3), (16, 2), (17, 24), (1, 64)])
@pytest.mark.parametrize("H,dv,rank", [(3, 128, 512), (2, 12, 200), (1, 16, 72), (2, 40, 36)])
def test_combine(R, S, H, dv, rank):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    RP = pad32(rank)
    part = torch.randn(R, H, S, RP, device="cuda") * torch.randn(R, H, S, 1, device="cuda").exp()
    ml = torch.rand(R, H, S, 2, device="cuda") * 5
    if S > 1:                                           # an empty split
        part[:, :, S // 2], ml[:, :, S // 2, 0], ml[:, :, S // 2, 1] = 0, -1e30, 0
    w = (torch.randn(H * dv, rank, device="cuda") * rank ** -0.5).bfloat16()
    got = hip_ops().latent_decode_combine(part, ml, w, dv)
    m, l = ml.double().unbind(-1)
    e = (m - m.amax(-1, keepdim=True)).exp()
    o = (part.double() * e[..., None]).sum(2) / (e * l).sum(-1)[..., None]
    wd = w.double().view(H, dv, rank)
    want = torch.stack([o[:, h, :rank] @ wd[h].t().contiguous() for h in range(H)], 1).reshape(R, -1)
    bf16_close(got, want)
    if S == 1:
        bf16_close(hip_ops().latent_decode_combine(part, None, w, dv),
                   torch.stack([part[:, h, 0, :rank].double() @ wd[h].t().contiguous()
                                for h in range(H)], 1).reshape(R, -1))


@pytest.mark.parametrize("R,H", [(63, 17), (64, 16), (64, 17), (65, 40), (64, 32)])
@pytest.mark.parametrize("rank,rot,splits", [(512, 64, 1), (512, 64, 3), (256, 32, 1), (128, 16, 2), (512, 128, 2)])
def test_attention_of_many_rows(R, H, rank, rot, splits):
    """Heads in pairs of tiles, two buffers of keys: from 64 rows and 17 heads on."""
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    RP, C, max_len = pad32(rank), pad32(rank) + pad32(rot), 330
    q = torch.randn(R, H, C, device="cuda").bfloat16()
    cache = torch.randn(R, max_len, C, device="cuda").bfloat16()
    pos = torch.randint(0, max_len, (R,), device="cuda", dtype=torch.int32)
    pos[:5] = torch.tensor([0, 63, 64, 127, max_len - 1])
    slot = torch.randperm(R, device="cuda").int()
    slot[7] = -1                                        # no sequence: zeros
    scale = C ** -0.5
    part, ml = hip_ops().latent_decode_attn(q, cache, slot, pos, rank, rot, scale, splits)
    assert (part[7] == 0).all() and (ml[7, ..., 1] == 0).all()
    m, l = ml.double().unbind(-1)
    e = (m - m.amax(-1, keepdim=True)).exp()
    got = (part.double() * e[..., None]).sum(2) / (e * l).sum(-1)[..., None]
    for r in range(R):
        if r != 7:
            keys = cache[slot[r], :pos[r] + 1].double()
            p = (q[r].double() @ keys.t().contiguous() * scale).softmax(-1)
            want = p @ keys[:, :RP]
            # probabilities are rounded to bf16 once
            assert (got[r] - want).norm() <= 2.0 ** -9 * 1.05 * (p @ keys[:, :RP].abs()).norm()
