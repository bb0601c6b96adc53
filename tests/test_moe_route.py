"""Device-side routing plan, the combine's backward and the two-pair dx."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (3, 2, 5), (64, 4, 64), (257, 8, 128), (1000, 6, 300), (40, 2, 4096),
                                   (9000, 8, 128), (33, 3, 1025)])
def test_route_plan(T, K, E):
    from automodel_amd.ops._backend import hip_ops

    g = torch.Generator().manual_seed(T)
    idx = torch.rand(T, E, generator=g).topk(K, -1)[1].cuda()
    probs = torch.rand(T, K, generator=g).cuda()
    counts, order, src, pos, perm_probs = hip_ops().route_plan(idx, probs, E)
    flat = idx.reshape(-1)
    want = flat.argsort(stable=True)
    assert torch.equal(order.long(), want)
    assert torch.equal(counts.long(), torch.bincount(flat, minlength=E))
    assert torch.equal(src.long(), want // K)
    assert torch.equal(pos.reshape(-1).long()[want], torch.arange(T * K, device="cuda"))
    assert torch.equal(perm_probs, probs.reshape(-1)[want])


@pytest.mark.parametrize("T,K,H", [(1, 1, 8), (37, 3, 520), (100, 8, 2048)])
def test_combine_backward(T, K, H):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    idx = torch.rand(T, 16).topk(K, -1)[1].cuda()
    probs = torch.rand(T, K, device="cuda")
    _, order, src, _, p = hip_ops().route_plan(idx, probs, 16)
    g = torch.randn(T, H, device="cuda").bfloat16()
    y = torch.randn(T * K, H, device="cuda").bfloat16()
    dy, dp = hip_ops().combine_bwd(g, y, src, order, p)
    gp = g.float()[src.long()]
    assert torch.equal(dy, (gp * p[:, None]).bfloat16())
    want = torch.empty(T * K, device="cuda", dtype=torch.float64)
    want[order.long()] = (gp.double() * y.double()).sum(-1)
    # H products summed in f32
    assert (dp.double() - want).abs().max() <= 2.0 ** -23 * H ** 0.5 * 4 * (gp.abs() * y.float().abs()).sum(-1).max()


@pytest.mark.parametrize("counts,N,K", [([5, 0, 130, 300], 128, 256), ([600, 0, 520], 1408, 128)])
@pytest.mark.parametrize("bm", [128, 256])
def test_two_pairs(counts, N, K, bm):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    M, E = sum(counts), len(counts)
    g1, g2 = (torch.randn(M, N, device="cuda").bfloat16() for _ in range(2))
    w1, w2 = (torch.randn(E, N, K, device="cuda").bfloat16() for _ in range(2))
    plan = hip_ops().build_group_plan(torch.tensor(counts, dtype=torch.int32, device="cuda"), M, bm)
    dx = hip_ops().grouped_gemm_nn2(g1, w1, g2, w2, *plan, bm)
    at = torch.tensor([0, *counts]).cumsum(0).tolist()
    want = torch.cat([g1[s].double() @ w1[e].double() + g2[s].double() @ w2[e].double()
                      for e, s in enumerate(slice(a, b) for a, b in zip(at, at[1:]))])
    assert (dx.double() - want).norm() <= 2.0 ** -9 * 1.02 * want.norm()
