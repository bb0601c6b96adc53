"""x w^T by csrc/linear_out.hip, and which calls it has (ops/linear.py: output_own, inferred)."""

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from automodel_amd.ops import linear as L

gpu = pytest.mark.gpu
cuda = pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")


def rand(*shape):
    return torch.randn(*shape, device="cuda").bfloat16()


def close(got, want, terms):
    # one rounding to 8 bits of each result, sums in 24 bits
    err = (got.double() - want).abs().max() / want.abs().max()
    assert got.shape == want.shape and err <= 2.0 ** -8 + terms * 2.0 ** -23, float(err)


# heights of 128 to 256, rows and columns that end within a tile, two steps and more, sums in parts with a short last one,
# more tiles than workgroups
@gpu
@cuda
@pytest.mark.parametrize("T,N,K,parts", [
    (1, 8, 128, False), (127, 264, 128, False), (129, 248, 192, False), (255, 1000, 320, False), (300, 520, 8256, True),
    (513, 1024, 8192, True), (700, 4096, 1408, None), (1025, 2816, 2048, None), (3003, 2816, 2048, False),
    (4100, 4104, 256, False), (257, 65544, 128, False),
])
def test_products(T, N, K, parts):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)
    x, w = rand(T, K), rand(N, K)
    height, cut = hip_ops().linear_y_cut(T, N, K)
    assert 128 <= height <= 256 and height % 32 == 0 and (parts is None or (cut > 1) == parts)
    want = x.double() @ w.double().t()
    close(hip_ops().linear_y(x, w), want, K)
    close(hip_ops().linear_y(x, w, True), want.relu().square(), K)


@gpu
@cuda
def test_squares_of_strange_sums():
    from automodel_amd.ops._backend import hip_ops

    for K in (128, 8256):
        x, w = torch.zeros(300, K, device="cuda").bfloat16(), rand(520, K).abs()
        x[1, 3], x[2, 5], x[3, 7], x[4, 9] = float("inf"), -float("inf"), float("nan"), -1e30
        y = hip_ops().linear_y(x, w, True)
        assert (y[1] == float("inf")).all() and (y[2] == 0).all() and y[3].isnan().all() and (y[4] == 0).all()
        assert (y[[0, 5, 299]] == 0).all()


@gpu
@cuda
@pytest.mark.parametrize("T,N,K", [(70, 72, 192), (300, 520, 8256)])
def test_edges_of_the_operands(T, N, K):
    """Nothing beyond an operand is read into a result: infinities behind its last row."""
    from automodel_amd.ops._backend import hip_ops

    def within(rows, cols):
        whole = torch.full((rows * cols + 65536,), float("inf"), device="cuda", dtype=torch.bfloat16)
        whole[: rows * cols] = torch.randn(rows * cols, device="cuda")
        return whole[: rows * cols].view(rows, cols)
    x, w = within(T, K), within(N, K)
    close(hip_ops().linear_y(x, w), x.double() @ w.double().t(), K)


@gpu
@cuda
def test_refusals():
    from automodel_amd.ops._backend import hip_ops

    y = hip_ops().linear_y
    for bad in (lambda: y(rand(4, 64), rand(8, 64)), lambda: y(rand(4, 160), rand(8, 160)), lambda: y(rand(4, 128), rand(12, 128)),
                lambda: y(rand(4, 128), rand(8, 192)), lambda: y(rand(4, 128).float(), rand(8, 128)),
                lambda: y(rand(128, 4).t(), rand(8, 128)), lambda: y(rand(1025)[1:].view(8, 128), rand(8, 128)),
                lambda: y(rand(8, 128).cpu(), rand(8, 128)), lambda: y(rand(128), rand(8, 128))):
        with pytest.raises(RuntimeError):
            bad()
    assert y(rand(0, 128), rand(8, 128)).shape == (0, 8)


def test_rule():
    assert L.output_own(3003, 2816, 2048) and L.output_own(511, 4096, 14336) and L.output_own(24000, 14336, 4096)
    # whole rounds of the library's tiles; few tiles; few rows
    for sizes in ((8192, 28672, 4096), (8192, 4096, 14336), (511, 4096, 4096), (255, 32768, 4096)):
        assert not L.output_own(*sizes)
    # few rows, where the weights' reads are the bound; a long sum in parts is another matter
    assert not L.output_own(384, 18432, 4096) and L.output_own(400, 18432, 4096) and L.output_own(384, 18432, 8192)
    # forms that the kernel refuses
    for sizes in ((3003, 2816, 2080), (3003, 2812, 2048), (65536, 4096, 64), (1 << 23, 4096, 128), (3000, 1 << 23, 128)):
        assert not L.output_own(*sizes)


@gpu
@cuda
@pytest.mark.parametrize("T,N,K", [(1001, 8256, 2112), (300, 4096, 8256), (200, 256, 512)])
def test_calls_without_gradients(T, N, K):
    from automodel_amd.ops._backend import hip_ops
    from automodel_amd.serving.decode_linear import DecodeLinear, project

    torch.manual_seed(0)
    lin = nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16)
    x = rand(T, K)
    own = hip_ops().small_nt if L.small(T, N, K) else hip_ops().linear_y
    with torch.no_grad():
        want = own(x, lin.weight)
        close(want, x.double() @ lin.weight.double().t(), K)
        for y in (L.linear(lin, x), DecodeLinear.from_linear(lin)(x), project(lin, x), L.inferred(x, lin.weight)):
            assert torch.equal(y, want) and not y.requires_grad
        assert torch.equal(L.linear(lin, x[None]), want[None])
        assert torch.equal(L.linear(lin, x, beside=True), F.linear(x, lin.weight))
        squares = project(lin, x, relu2=True)
        if not L.squared_own(T, N, K):             # a pass of its own, over rounded results
            assert torch.equal(squares, F.relu(want.float()).square().bfloat16())
        else:
            close(squares, (x.double() @ lin.weight.double().t()).relu().square(), K)
        # what the kernels do not take is the library's, as before
        strange = (rand(T, 2 * K)[:, ::2], rand(T * K + 1)[1:].view(T, K), rand(K, T).t(), rand(1, K).expand(T, K))
        for v in strange:
            assert L.inferred(v, lin.weight) is None and torch.equal(L.linear(lin, v), F.linear(v, lin.weight))
        assert L.inferred(x.float(), lin.weight.float()) is None and L.inferred(x[:0], lin.weight) is None
        assert L.inferred(x.cpu(), lin.weight.cpu()) is None
        with torch.autocast("cuda", dtype=torch.float16):
            assert L.linear(lin, x).dtype == torch.float16
        biased = nn.Linear(K, N, device="cuda", dtype=torch.bfloat16)
        assert torch.equal(L.linear(biased, x), F.linear(x, biased.weight, biased.bias))
        seen = []
        hook = lin.register_forward_hook(lambda *_: seen.append(1))
        L.linear(lin, x)
        hook.remove()
        assert seen
    assert L.inferred(x, lin.weight) is None       # gradients may be wanted
    assert torch.equal(torch.func.vmap(lambda v: L.linear(lin, v))(x[None])[0].detach(), F.linear(x, lin.weight).detach())


@gpu
@cuda
def test_layer_in_training():
    torch.manual_seed(0)
    T, N, K = 1001, 8256, 2112
    lin = nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16)
    x, g = rand(7, T // 7, K).requires_grad_(), rand(7, T // 7, N)
    y = L.linear(lin, x)
    close(y, x.double() @ lin.weight.double().t(), K)
    dx, dw = torch.autograd.grad(y, (x, lin.weight), g)
    close(dx, g.double() @ lin.weight.double(), N)
    close(dw, g.flatten(0, 1).double().t() @ x.flatten(0, 1).double(), T)
    assert torch.equal(L.linear(lin, x, beside=True), F.linear(x, lin.weight))
    strange = x.detach().transpose(0, 1).contiguous().transpose(0, 1)
    close(L.linear(lin, strange), y.double(), K)
