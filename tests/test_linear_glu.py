"""silu(x w^T) (x up^T) in one kernel (csrc/linear_out.hip: linear_glu), and which calls it has."""

import pytest
import torch
import torch.nn as nn

from automodel_amd.ops import linear as L

gpu = pytest.mark.gpu
cuda = pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")


def rand(*shape, std=1.0):
    return (torch.randn(*shape, device="cuda") * std).bfloat16()


def reference(x, w, up):
    a, b = x.double() @ w.double().t(), x.double() @ up.double().t()
    return a * torch.sigmoid(a) * b


# one row, every height of a tile, a part of 16 columns, of a wave's 64, of a tile's 128; more tiles than workgroups
@gpu
@cuda
@pytest.mark.parametrize("T,I,K", [(1, 8, 128), (127, 72, 192), (129, 136, 128), (200, 520, 2048), (300, 1000, 512),
                                   (700, 2816, 1024), (1025, 1544, 2112), (4100, 2056, 128), (257, 32776, 128)])
def test_products(T, I, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)
    x, w, up = rand(T, K), rand(I, K, std=K ** -0.5), rand(I, K, std=K ** -0.5)
    got, want = hip_ops().linear_glu(x, w, up), reference(x, w, up)
    # one rounding to 8 bits of results, whose sums, exponential and quotient have 20 at least; 2^-8 of each result at
    # most, half of that in the mean of many
    assert got.shape == want.shape
    assert (got.double() - want).norm() <= 2.0 ** (-9 if T > 1 else -8) * 1.05 * want.norm()
    err = (got.double() - want).abs() - 2.0 ** -8 * want.abs()
    assert err.max() <= 2.0 ** -20 * K ** 0.5 * want.abs().max()


@gpu
@cuda
def test_edges_and_strange_sums():
    from automodel_amd.ops._backend import hip_ops

    def within(v):
        whole = torch.full((v.numel() + 65536,), float("inf"), device="cuda", dtype=torch.bfloat16)
        whole[: v.numel()] = v.flatten()
        return whole[: v.numel()].view(v.shape)
    torch.manual_seed(0)
    x, w, up = within(rand(70, 192)), within(rand(72, 192, std=0.1)), within(rand(72, 192, std=0.1))
    got, want = hip_ops().linear_glu(x, w, up), reference(x, w, up)
    assert (got.double() - want).norm() <= 2.0 ** -9 * 1.05 * want.norm()
    x, w, up = torch.zeros(8, 128, device="cuda").bfloat16(), rand(64, 128).abs() + 1, rand(64, 128).abs() + 1
    x[0, 0], x[1, 0], x[2, 0], x[3, 0], x[4, 0] = float("inf"), float("nan"), -500.0, 500.0, -float("inf")
    y = hip_ops().linear_glu(x, w, up)
    assert (y[0] == float("inf")).all() and y[1].isnan().all() and y[4].isnan().all()      # as silu(-inf) has it
    assert (y[2] == 0).all() and (y[3] > 0).all() and y[3].isfinite().all() and (y[5:] == 0).all()


@gpu
@cuda
def test_refusals():
    from automodel_amd.ops._backend import hip_ops

    op = hip_ops().linear_glu
    for bad in ((rand(4, 64), rand(8, 64), rand(8, 64)), (rand(4, 160), rand(8, 160), rand(8, 160)),
                (rand(4, 128), rand(12, 128), rand(12, 128)), (rand(4, 128), rand(8, 128), rand(16, 128)),
                (rand(4, 128), rand(8, 128), rand(128, 8).t()), (rand(4, 128), rand(8, 128), rand(8, 128).cpu()),
                (rand(4, 128), rand(8, 128), rand(1025)[1:].view(8, 128)), (rand(4, 128), rand(8, 128), rand(8, 128).float()),
                (rand(4, 192), rand(8, 128), rand(8, 128))):
        with pytest.raises(RuntimeError):
            op(*bad)
    assert op(rand(0, 128), rand(8, 128), rand(8, 128)).shape == (0, 8)


def test_rule():
    assert L.gated_own(511, 14336, 4096) and L.gated_own(8192, 14336, 4096) and L.gated_own(600, 1024, 1024)
    for sizes in ((128, 14336, 4096), (511, 4096, 4096), (200, 4096, 2048), (511, 14336, 4128), (511, 14340, 4096),
                  (1 << 23, 4096, 128)):
        assert not L.gated_own(*sizes)


@gpu
@cuda
@pytest.mark.parametrize("fused", [False, True])
def test_layers(fused):
    from automodel_amd.ops.swiglu import swiglu
    from automodel_amd.serving.decode_linear import DecodeLinear, glu_rows

    torch.manual_seed(0)
    T, I, K = 600, 1024, 512
    lins = [nn.Linear(K, 2 * I if fused else I, bias=False, device="cuda", dtype=torch.bfloat16) for _ in range(1 if fused else 2)]
    w, up = lins[0].weight.chunk(2) if fused else [lin.weight for lin in lins]
    x = rand(2, T // 2, K)
    want = reference(x, w, up)
    assert glu_rows(lins, x) is None                  # gradients may be wanted
    with torch.no_grad():
        for ls in (lins, [DecodeLinear.from_linear(lin) for lin in lins]):
            y = glu_rows(ls, x)
            assert y.shape == want.shape and (y.double() - want).norm() <= 2.0 ** -9 * 1.05 * want.norm()
        ref = swiglu(x @ w.t(), x @ up.t())
        assert (y.double() - want).norm() <= (ref.double() - want).norm()
        for strange in (x.transpose(0, 1), x[:, :10], rand(T * K + 1)[1:].view(2, T // 2, K), x.float(), x.cpu()):
            assert glu_rows(lins, strange) is None
        biased = [nn.Linear(K, lin.out_features, device="cuda", dtype=torch.bfloat16) for lin in lins]
        assert glu_rows(biased, x) is None
        hook = lins[0].register_forward_hook(lambda *_: None)
        assert glu_rows(lins, x) is None
        hook.remove()
        with torch.autocast("cuda", dtype=torch.float16):
            assert glu_rows(lins, x) is None
