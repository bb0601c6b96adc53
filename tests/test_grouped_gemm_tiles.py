"""Grouped GEMM at the edges of its tiles: empty and one-row groups, widths that are no
multiple of a tile, both row tiles, against f64."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("counts,N,K", [
    ([5, 0, 130, 128, 1, 300], 128, 64), ([64, 64], 256, 128), ([0, 0, 7], 384, 192),
    ([257, 3, 0, 511], 1408, 128), ([1000], 128, 1408), ([129] * 9, 256, 320), ([0, 0], 128, 128),
    ([1] * 300, 128, 128),
])
@pytest.mark.parametrize("bm", [128, 256])
def test_grouped_gemm(counts, N, K, bm):
    from automodel_amd.ops._backend import hip_ops

    ops = hip_ops()
    torch.manual_seed(0)
    M, E = sum(counts), len(counts)
    x = torch.randn(M, K, device="cuda").bfloat16()
    g = torch.randn(M, N, device="cuda").bfloat16()
    w = torch.randn(E, N, K, device="cuda").bfloat16()
    offs, tile_map, n_tiles = ops.build_group_plan(
        torch.tensor(counts, dtype=torch.int32, device="cuda"), M, bm)
    at = torch.tensor([0, *counts]).cumsum(0).tolist()
    assert offs.tolist() == at
    assert tile_map[: int(n_tiles)].tolist() == [
        [e, at[e] + m] for e in range(E) for m in range(0, counts[e], bm)]

    def close(got, want):       # f32 sums, rounded to bf16 once
        assert (got.double() - want).norm() <= 2.0 ** -9 * 1.02 * want.norm()

    part = [slice(at[e], at[e + 1]) for e in range(E)]
    close(ops.grouped_gemm_nt(x, w, offs, tile_map, n_tiles, bm),
          torch.cat([x[s].double() @ w[e].double().t() for e, s in enumerate(part)]))
    if K % 128 == 0:
        close(ops.grouped_gemm_nn(g, w, offs, tile_map, n_tiles, bm),
              torch.cat([g[s].double() @ w[e].double() for e, s in enumerate(part)]))
        close(ops.grouped_gemm_tn(g, x, offs, E),
              torch.stack([g[s].double().t() @ x[s].double() for s in part]))


# rows of 512 per group and more on average: the weight gradients' 256 x 256 tiles of four waves
@pytest.mark.parametrize("counts,N,K", [
    ([1600, 0, 31, 513], 384, 640), ([1, 1, 2000], 128, 128), ([512, 512], 256, 1408),
    ([0, 0, 3000], 128, 384), ([2000, 33, 1], 896, 256), ([1025], 128, 128), ([1535, 1], 128, 128),
])
def test_grouped_weight_gradient(counts, N, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)

    def close(got, want):       # f32 sums, rounded to bf16 once
        assert (got.double() - want).norm() <= 2.0 ** -9 * 1.02 * want.norm()

    M, E = sum(counts), len(counts)
    assert M >= 512 * E
    g, x = (torch.randn(M, n, device="cuda").bfloat16() for n in (N, K))
    at = torch.tensor([0, *counts]).cumsum(0).tolist()
    part = [slice(at[e], at[e + 1]) for e in range(E)]
    offs = torch.tensor(at, dtype=torch.int32, device="cuda")
    want = torch.stack([g[s].double().t() @ x[s].double() for s in part])
    close(hip_ops().grouped_gemm_tn(g, x, offs, E), want)
    # a group's infinities stay its own
    for e in range(E):
        if counts[e]:
            gi, xi = g.clone(), x.clone()
            gi[part[e]], xi[part[e]] = float("inf"), float("inf")
            got = hip_ops().grouped_gemm_tn(gi, xi, offs, E)
            rest = [i for i in range(E) if i != e]
            assert not got[e].isfinite().any()
            if rest and want[rest].norm() > 0:
                close(got[rest], want[rest])


UNEVEN = [1, 129, 160, 161, 0, 193, 225, 256, 257, 300, 33, 400, 513, 1030, 3000, 2100, 32]


# Tiles of 4 to 8 times 32 rows, dealt to workgroups that stay: tall and short ones, one part and several, fewer tiles than
# workgroups and more, tables of more than a wave's groups and more groups than they hold
@pytest.mark.parametrize("counts,N,K,caps", [
    (UNEVEN, 640, 640, (256, 256, 256)), (UNEVEN, 128, 576, (128, None, None)), ([700], 512, 256, (128, 128, 256)),
    (UNEVEN, 3456, 512, (256, 128, 256)), (UNEVEN, 512, 3456, (128, 256, 256)), (UNEVEN, 128, 3456, (128, 0, 256)),
    ([1600, 0, 31, 513], 3456, 512, (256, 128, 256)), ([512] * 6 + [3000], 1408, 1408, (256, 256, 256)),
    ([130, 250, 200, 255] * 16, 768, 768, (256, 256, 256)), ([90, 110] * 20, 1024, 256, (0, 128, 0)),
    ([40, 1000] * 120, 512, 512, (256, 256, 256)), ([30, 990] * 150, 1152, 1024, (256, 256, 256)),
    ([40] * 513, 1152, 1024, (0, 0, 0)),
])
def test_tiles_of_unequal_heights(counts, N, K, caps):
    from automodel_amd.ops._backend import hip_ops

    ops = hip_ops()
    torch.manual_seed(1)
    M, E = sum(counts), len(counts)
    assert all(c is None or ops.grouped_gemm_cap(m, M, E, N, K) == c for m, c in enumerate(caps))
    x, g, g2 = (torch.randn(M, n, device="cuda").bfloat16() for n in (K, N, N))
    w, w2 = (torch.randn(E, N, K, device="cuda").bfloat16() for _ in range(2))
    bm = 256 if M >= 512 * E else 128
    plan = (*ops.build_group_plan(torch.tensor(counts, dtype=torch.int32, device="cuda"), M, bm), bm)
    at = torch.tensor([0, *counts]).cumsum(0).tolist()
    part = [slice(at[e], at[e + 1]) for e in range(E)]

    def close(got, want):       # f32 sums, rounded to bf16 once
        assert (got.double() - want).norm() <= 2.0 ** -9 * 1.02 * want.norm()

    nt = torch.cat([x[s].double() @ w[e].double().t() for e, s in enumerate(part)])
    close(ops.grouped_gemm_nt(x, w, *plan), nt)
    if K % 128 == 0:
        nn = torch.cat([g[s].double() @ w[e].double() for e, s in enumerate(part)])
        close(ops.grouped_gemm_nn(g, w, *plan), nn)
        nn += torch.cat([g2[s].double() @ w2[e].double() for e, s in enumerate(part)])
        close(ops.grouped_gemm_nn2(g, w, g2, w2, *plan), nn)
        tn = torch.stack([g[s].double().t() @ x[s].double() for s in part])
        close(ops.grouped_gemm_tn(g, x, plan[0], E), tn)
        # a group's infinities stay its own
        e = max(range(E), key=lambda i: counts[i])
        gi, xi = g.clone(), x.clone()
        gi[part[e]], xi[part[e]] = float("inf"), float("inf")
        own = torch.zeros(M, dtype=torch.bool, device="cuda")
        own[part[e]] = True
        close(ops.grouped_gemm_nt(xi, w, *plan)[~own], nt[~own])
        assert ops.grouped_gemm_nn(gi, w, *plan)[~own].isfinite().all()
        got = ops.grouped_gemm_tn(gi, xi, plan[0], E)
        close(torch.cat([got[:e], got[e + 1:]]), torch.cat([tn[:e], tn[e + 1:]]))


def test_more_tiles_than_are_dealt_out():
    from automodel_amd.ops._backend import hip_ops

    ops = hip_ops()
    torch.manual_seed(2)
    M, N, K = 65000, 16384, 512            # 254 x 64 tiles, more than 48 for each of 256 workgroups
    x, w = torch.randn(M, K, device="cuda").bfloat16(), torch.randn(1, N, K, device="cuda").bfloat16()
    assert ops.grouped_gemm_cap(0, M, 1, N, K) == 256
    plan = ops.build_group_plan(torch.tensor([M], dtype=torch.int32, device="cuda"), M, 256)
    got = ops.grouped_gemm_nt(x, w, *plan, 256)
    rows = torch.cat([torch.randperm(M, device="cuda")[:1000], torch.tensor([0, M - 1], device="cuda")])
    want = x[rows].double() @ w[0].double().t()
    assert (got[rows].double() - want).norm() <= 2.0 ** -9 * 1.02 * want.norm()
    for i in range(0, M, 8192):            # every tile is there
        assert (got[i:i + 8192].abs().amax(1) > 0).all()


@pytest.mark.parametrize("E,rows,N,K,caps", [
    (64, 1000, 128, 2048, (0, 0, 256)), (64, 1000, 2048, 128, (0, 0, 0)),       # half a tile's columns
    (64, 1000, 384, 2048, (256, 0, 256)), (64, 1000, 2048, 384, (0, 256, 256)),     # short sums
    (8, 700, 1024, 256, (128, 128, 256)), (8, 700, 256, 128, (0, 0, 0)),        # in few tiles
    (256, 191, 512, 256, (0, 0, 0)), (256, 400, 512, 512, (256, 256, 256)),     # many groups
    (400, 400, 512, 512, (0, 0, 0)), (400, 300, 1408, 2048, (256, 256, 256)), (513, 400, 1408, 2048, (0, 0, 0)),
    (64, 150, 768, 2048, (0, 256, 256)), (64, 100, 768, 1024, (0, 0, 0)),       # few rows
])
def test_rule(E, rows, N, K, caps):
    from automodel_amd.ops._backend import hip_ops

    assert tuple(hip_ops().grouped_gemm_cap(m, E * rows, E, N, K) for m in range(3)) == caps
