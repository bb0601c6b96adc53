"""Gate, up and their activation of grouped experts in one kernel (csrc/grouped_gemm.hip: grouped_glu)."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def rand(*shape, std=1.0):
    return (torch.randn(*shape, device="cuda") * std).bfloat16()


def plan(counts):
    from automodel_amd.ops._backend import hip_ops

    return (*hip_ops().build_group_plan(torch.tensor(counts, device="cuda", dtype=torch.int32), sum(counts), 128), 128)


# groups of none, one and several tiles with remainders, one column tile and a cut one, the kernel by the plan and the other
@pytest.mark.parametrize("counts,N,K,tiles", [
    ([600, 0, 1, 500, 129, 2000, 257, 1000], 768, 2048, True), ([5000], 384, 512, True), ([1300, 1024, 900, 1100], 1408, 1024, True),
    ([700] * 16, 256, 512, True), ([513] * 40, 640, 512, True), ([20, 0, 3, 60], 256, 128, False), ([64] * 8, 128, 512, False),
])
def test_products(counts, N, K, tiles):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(N)
    ops, M, E = hip_ops(), sum(counts), len(counts)
    x, w, up = rand(M, K), rand(E, N, K, std=K ** -0.5), rand(E, N, K, std=K ** -0.5)
    p = plan(counts)
    assert (ops.grouped_gemm_cap(0, M, E, 2 * N, K) > 0) == tiles
    g, u, h = ops.grouped_glu(x, w, up, *p)
    parts = list(zip(x.split(counts), w, up))
    a, b = (torch.cat([v[0].double() @ v[i].double().t() for v in parts]) for i in (1, 2))
    for got, ref in ((g, a), (u, b)):                 # one rounding to 8 bits each
        assert got.shape == ref.shape and (got.double() - ref).norm() <= 2.0 ** -9 * 1.05 * ref.norm()
    assert torch.equal(g, ops.grouped_gemm_nt(x, w, *p)) and torch.equal(u, ops.grouped_gemm_nt(x, up, *p))
    assert torch.equal(h, ops.swiglu_fwd(g, u))


def test_strange_sums():
    from automodel_amd.ops._backend import hip_ops

    ops, M, N, K = hip_ops(), 4096, 256, 512
    x, w, up = torch.zeros(M, K, device="cuda").bfloat16(), rand(1, N, K).abs() + 1, rand(1, N, K).abs() + 1
    for i, v in enumerate((float("inf"), float("nan"), -500.0, 500.0, -float("inf"), -20.0, 1e-30)):
        x[i, 0] = v
    assert ops.grouped_gemm_cap(0, M, 1, 2 * N, K) > 0
    g, u, h = ops.grouped_glu(x, w, up, *plan([M]))
    want = ops.swiglu_fwd(g, u)
    assert torch.equal(h.isnan(), want.isnan()) and torch.equal(h.nan_to_num(), want.nan_to_num())


def test_operands_of_other_forms():
    from automodel_amd.ops._backend import hip_ops

    ops, counts, N, K = hip_ops(), [700, 900], 256, 512
    M, p = sum(counts), plan(counts)
    x, w, up = rand(M, K), rand(2, N, K), rand(2, N, K)
    for bad in ((x, w, up[:1]), (x, w, up.float()), (x, w, up.transpose(1, 2).contiguous().transpose(1, 2)), (x, w, up.cpu()),
                (x[:, :256], w, up), (x.float(), w, up)):
        with pytest.raises(RuntimeError):
            ops.grouped_glu(*bad, *p)
    off = rand(M * K + 1)[1:].view(M, K)               # not at 16 bytes: the kernel before
    for got, ref in zip(ops.grouped_glu(off, w, up, *p), ops.grouped_glu(off.clone(), w, up, *p)):
        assert (got.double() - ref.double()).norm() <= 2.0 ** -7 * ref.double().norm()
    assert ops.grouped_glu(x[:0], w, up, *plan([0, 0]))[2].shape == (0, N)
