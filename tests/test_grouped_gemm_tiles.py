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
