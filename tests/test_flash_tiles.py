"""Flash attention at the edges of its tiles, against plain f32 attention."""

import math

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def _reference(q, k, v, causal, q_start, doc_start, scale):
    G = q.shape[2] // k.shape[2]
    q, k, v = (t.float().transpose(1, 2) for t in (q, k, v))
    k, v = (t.repeat_interleave(G, 1) for t in (k, v))
    s = (q @ k.transpose(-1, -2).contiguous()) * scale
    qpos = torch.arange(q_start, q_start + q.shape[2], device="cuda")[:, None]
    kpos = torch.arange(k.shape[2], device="cuda")[None]
    keep = (kpos <= qpos) if causal else torch.ones_like(kpos <= qpos)
    if doc_start is not None:
        keep = keep & (kpos >= doc_start[qpos])
    s = s.masked_fill(~keep, -math.inf)
    return (s.softmax(-1) @ v).transpose(1, 2), s.logsumexp(-1)


def _docs(cuts, total):
    start = torch.empty(total, dtype=torch.int32)
    end = torch.empty(total, dtype=torch.int32)
    for a, b in zip([0, *cuts], [*cuts, total]):
        start[a:b], end[a:b] = a, b
    return start.cuda(), end.cuda()


def _grads(fn, args, dout):
    args = [t.detach().clone().requires_grad_() for t in args]
    return torch.autograd.grad(fn(*args), args, dout)


# probabilities and the output are each rounded to bf16 once (2^-9 of a value at most)
FWD = 2 * 2.0 ** -9


@pytest.mark.parametrize("dims", [(64, 64), (96, 96), (128, 128), (192, 128), (192, 192), (256, 256)])
@pytest.mark.parametrize("sq,skv,causal,q_start,cuts,scale", [
    (128, 128, True, 0, None, 1.0),
    (384, 352, False, 0, None, 1.0),            # last tile half empty, three blocks
    (256, 640, True, 384, None, 1.0),           # a chunk behind a prefix
    (640, 640, True, 0, (1, 63, 64, 65, 130, 500), 1.0),
    (256, 768, True, 256, (100, 300, 301), 1.0),
    (256, 256, True, 0, None, -1.0),
    (256, 256, True, 0, None, 0.0),
    (1, 1, True, 0, None, 1.0),
    (129, 129, True, 0, None, 1.0),
    (333, 333, True, 0, (5, 200, 201), 1.0),
])
def test_forward(dims, sq, skv, causal, q_start, cuts, scale):
    torch.manual_seed(0)
    q = torch.randn(1, sq, 4, dims[0], device="cuda").bfloat16() * 2
    k = torch.randn(1, skv, 2, dims[0], device="cuda").bfloat16()
    v = torch.randn(1, skv, 2, dims[1], device="cuda").bfloat16()
    k[:, skv // 3] *= 8                         # scores that stand out: the maximum moves
    scale *= dims[0] ** -0.5
    start = None if cuts is None else _docs(cuts, skv)[0]
    from automodel_amd.ops._backend import hip_ops

    o, lse = hip_ops().flash_attn_fwd(q, k, v, scale, causal, q_start, start)
    ro, rlse = _reference(q, k, v, causal, q_start, start, scale)
    assert (o.float() - ro).norm() / ro.norm() < FWD
    assert (lse - rlse).abs().max() < 1e-5 * max(1.0, float(rlse.abs().max()))


@pytest.mark.parametrize("dims", [(64, 64), (128, 128), (192, 128), (256, 256)])
@pytest.mark.parametrize("s,causal,cuts", [(160, True, None), (544, True, None), (701, False, None),
                                           (832, False, None), (448, True, ()), (1344, True, (40, 1000))])
def test_last_tiles_without_a_successor(dims, s, causal, cuts):
    """Waves whose whole tiles reach up to the last one but one."""
    torch.manual_seed(0)
    q = torch.randn(1, s, 4, dims[0], device="cuda").bfloat16()
    k = torch.randn(1, s, 2, dims[0], device="cuda").bfloat16()
    v = torch.randn(1, s, 2, dims[1], device="cuda").bfloat16()
    start = None if cuts is None else _docs(cuts, s)[0]
    from automodel_amd.ops._backend import hip_ops

    o, _ = hip_ops().flash_attn_fwd(q, k, v, dims[0] ** -0.5, causal, 0, start)
    ro, _ = _reference(q, k, v, causal, 0, start, dims[0] ** -0.5)
    assert (o.float() - ro).norm() / ro.norm() < FWD


# dS is rounded to bf16 once and so is each gradient; P and the delta of a bf16 output bring
# about the same again
BWD = 4 * 2.0 ** -9


@pytest.mark.parametrize("dims", [(64, 64), (96, 96), (128, 128), (192, 128), (192, 192), (256, 256)])
@pytest.mark.parametrize("sq,skv,causal,q_start,cuts,scale", [
    (128, 128, True, 0, None, 1.0),
    (384, 256, False, 0, None, 1.0),
    (256, 640, True, 384, None, 1.0),
    (640, 640, True, 0, (1, 63, 64, 65, 130, 500), 1.0),
    (256, 768, True, 256, (100, 300, 301), 1.0),
    (256, 256, True, 0, None, -1.0),
    (17, 17, True, 0, None, 1.0),
    (129, 129, True, 0, None, 1.0),
    (333, 333, True, 0, (5, 200, 201), 1.0),
])
def test_backward(dims, sq, skv, causal, q_start, cuts, scale):
    torch.manual_seed(0)
    q = torch.randn(2 if cuts is None else 1, sq, 4, dims[0], device="cuda").bfloat16()
    k = torch.randn(q.shape[0], skv, 2, dims[0], device="cuda").bfloat16()
    v = torch.randn(q.shape[0], skv, 2, dims[1], device="cuda").bfloat16()
    do = torch.randn(q.shape[0], sq, 4, dims[1], device="cuda").bfloat16()
    scale *= dims[0] ** -0.5
    start, end = (None, None) if cuts is None else _docs(cuts, skv)
    from automodel_amd.ops.attention import _FlashAttnHip

    got = _grads(lambda *t: _FlashAttnHip.apply(*t, causal, scale, q_start, start, end), (q, k, v), do)
    ref = _grads(lambda *t: _reference(*t, causal, q_start, start, scale)[0],
                 (q.float(), k.float(), v.float()), do.float())
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        assert (g.float() - r).norm() / r.norm() < BWD, name


# dK and dV walk the tiles of all heads of a group from the last one on, four (128) or three
# (192, 128) buffers in turn: fewer tiles than buffers, several rounds of them, short last tiles,
# groups of one head and of four
@pytest.mark.parametrize("dims", [(128, 128), (192, 128)])
@pytest.mark.parametrize("heads", [(2, 2), (8, 2)])
@pytest.mark.parametrize("sq,skv,causal,q_start,cuts", [
    (64, 64, False, 0, None), (65, 65, True, 0, None), (200, 333, False, 0, None),
    (1000, 1000, True, 0, None), (700, 1211, True, 511, None), (1088, 1088, True, 0, (300, 301, 650, 1000)),
])
def test_key_gradients_over_many_tiles(dims, heads, sq, skv, causal, q_start, cuts):
    torch.manual_seed(0)
    B = 2 if cuts is None else 1
    q = torch.randn(B, sq, heads[0], dims[0], device="cuda").bfloat16()
    k = torch.randn(B, skv, heads[1], dims[0], device="cuda").bfloat16()
    v = torch.randn(B, skv, heads[1], dims[1], device="cuda").bfloat16()
    do = torch.randn(B, sq, heads[0], dims[1], device="cuda").bfloat16()
    scale = dims[0] ** -0.5
    start, end = (None, None) if cuts is None else _docs(cuts, skv)
    from automodel_amd.ops.attention import _FlashAttnHip

    run = lambda: _grads(lambda *t: _FlashAttnHip.apply(*t, causal, scale, q_start, start, end), (q, k, v), do)
    got = run()
    ref = _grads(lambda *t: _reference(*t, causal, q_start, start, scale)[0],
                 (q.float(), k.float(), v.float()), do.float())
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        assert (g.float() - r).norm() / r.norm() < BWD, name
    for first, again in zip(got, run()):        # the same bits
        assert torch.equal(first, again)


# dQ of long walks, three buffers in turn: workgroups of 256 (192 for keys of 192) rows of which the last
# is short, short last key tiles, a diagonal that ends some waves of a workgroup early
@pytest.mark.parametrize("dims", [(128, 128), (192, 128)])
@pytest.mark.parametrize("B,heads,sq,skv,causal,q_start", [
    (4, (32, 32), 257, 1024, False, 0), (4, (48, 16), 300, 1100, True, 800), (4, (32, 32), 200, 1281, True, 1081),
    (3, (32, 8), 1030, 1030, True, 0), (1, (16, 16), 1, 1024, True, 1023),
])
def test_query_gradients_of_long_walks(dims, B, heads, sq, skv, causal, q_start):
    torch.manual_seed(0)
    q = torch.randn(B, sq, heads[0], dims[0], device="cuda").bfloat16()
    k = torch.randn(B, skv, heads[1], dims[0], device="cuda").bfloat16()
    v = torch.randn(B, skv, heads[1], dims[1], device="cuda").bfloat16()
    do = torch.randn(B, sq, heads[0], dims[1], device="cuda").bfloat16()
    scale = dims[0] ** -0.5
    from automodel_amd.ops.attention import _FlashAttnHip

    run = lambda: _grads(lambda *t: _FlashAttnHip.apply(*t, causal, scale, q_start, None, None), (q, k, v), do)
    got = run()
    for b in range(B):              # (the reference holds a score for every pair)
        ref = _grads(lambda *t: _reference(*t, causal, q_start, None, scale)[0],
                     [t[b : b + 1].float() for t in (q, k, v)], do[b : b + 1].float())
        for name, g, r in zip(("dq", "dk", "dv"), got, ref):
            assert (g[b : b + 1].float() - r).norm() / r.norm() < BWD, name
    for first, again in zip(got, run()):        # the same bits
        assert torch.equal(first, again)


# packed rows of short documents have another backward where their number is known
@pytest.mark.parametrize("dims", [(128, 128), (192, 128)])
@pytest.mark.parametrize("heads,sq,q_start,step", [((4, 2), 640, 0, 64), ((4, 4), 333, 0, 37), ((2, 2), 256, 256, 31)])
def test_short_documents(dims, heads, sq, q_start, step):
    from automodel_amd.ops._backend import hip_ops
    from automodel_amd.ops.attention import _FlashAttnHip

    torch.manual_seed(0)
    skv = sq + q_start
    cuts = tuple(range(step, skv, step))
    start, end = _docs(cuts, skv)
    q = torch.randn(1, sq, heads[0], dims[0], device="cuda").bfloat16()
    k = torch.randn(1, skv, heads[1], dims[0], device="cuda").bfloat16()
    v = torch.randn(1, skv, heads[1], dims[1], device="cuda").bfloat16()
    do = torch.randn(1, sq, heads[0], dims[1], device="cuda").bfloat16()
    scale, docs = dims[0] ** -0.5, len(cuts) + 1
    assert not hip_ops().flash_attn_bwd_ordered(1, sq, skv, *heads, *dims, True, docs)[0]
    got = _grads(lambda *t: _FlashAttnHip.apply(*t, True, scale, q_start, start, end, docs), (q, k, v), do)
    ref = _grads(lambda *t: _reference(*t, True, q_start, start, scale)[0],
                 (q.float(), k.float(), v.float()), do.float())
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        assert (g.float() - r).norm() / r.norm() < BWD, name


def test_document_bounds():
    from automodel_amd.ops.attention import doc_bounds_from_cu

    for cu, total in ([0, 3, 3, 7, 300], 300), ([0, 5, 260], 301), ([0, 1], 1):
        cu = torch.tensor(cu, dtype=torch.int32)
        for got, want in zip(doc_bounds_from_cu(cu.cuda(), total), doc_bounds_from_cu(cu, total)):
            assert got.dtype == want.dtype and torch.equal(got.cpu(), want)
