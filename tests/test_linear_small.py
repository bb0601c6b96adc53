"""Products of small layers (csrc/linear_small.hip) and the node of autograd around them (csrc/linear_node.cpp)."""

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


# tiles' edges and remainders, sums below a step, of several and in parts of both sizes of tile; one row, 8 columns
@gpu
@cuda
@pytest.mark.parametrize("T,N,K", [
    (1, 8, 8), (1, 64, 64), (63, 72, 136), (65, 64, 128), (200, 1000, 520), (513, 264, 328), (129, 8, 4096),
    (7, 128, 4096), (256, 256, 256), (1025, 1536, 1544), (4096, 512, 512), (2000, 200, 64),
])
def test_products(T, N, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)
    ops, x, w, g = hip_ops(), rand(T, K), rand(N, K), rand(T, N)
    close(ops.small_nt(x, w), x.double() @ w.double().t(), K)
    close(ops.small_nn(g, w), g.double() @ w.double(), N)
    close(ops.small_tn(g, x), g.double().t() @ x.double(), T)


# both sides of the line between the kernels of few rows and of tiles; whole and broken steps of either
@gpu
@cuda
@pytest.mark.parametrize("T", [2, 15, 16, 17])
@pytest.mark.parametrize("N,K", [(8, 4104), (72, 136), (1000, 512), (1536, 64)])
def test_few_rows(T, N, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)

    def within(*shape):                  # nothing beyond an operand is read into a result
        whole = torch.full((shape[0] * shape[1] + 4096,), float("inf"), device="cuda", dtype=torch.bfloat16)
        whole[: shape[0] * shape[1]] = torch.randn(shape[0] * shape[1], device="cuda")
        return whole[: shape[0] * shape[1]].view(shape)
    x, w = within(T, K), within(N, K)
    close(hip_ops().small_nt(x, w), x.double() @ w.double().t(), K)


@gpu
@cuda
def test_edges_of_the_operands():
    """Nothing beyond an operand is read into a result: infinities behind its last row and column."""
    from automodel_amd.ops._backend import hip_ops

    ops, T, N, K = hip_ops(), 70, 72, 40
    for mode, (r, c) in enumerate((((T, K), (N, K)), ((T, N), (N, K)), ((T, N), (T, K)))):
        def within(shape):
            whole = torch.full((shape[0] * shape[1] + 4096,), float("inf"), device="cuda", dtype=torch.bfloat16)
            whole[: shape[0] * shape[1]] = torch.randn(shape[0] * shape[1], device="cuda")
            return whole[: shape[0] * shape[1]].view(shape)
        a, b = within(r), within(c)
        p, q = a.double(), b.double()
        want = (lambda: p @ q.t(), lambda: p @ q, lambda: p.t() @ q)[mode]()
        close((ops.small_nt, ops.small_nn, ops.small_tn)[mode](a, b), want, 100)


@gpu
@cuda
def test_refusals_and_cuts():
    from automodel_amd.ops._backend import hip_ops

    ops = hip_ops()
    for bad in (lambda: ops.small_nt(rand(4, 12), rand(8, 12)), lambda: ops.small_nt(rand(4, 8), rand(12, 8)),
                lambda: ops.small_nt(rand(4, 8), rand(8, 16)), lambda: ops.small_nn(rand(4, 8), rand(16, 8)),
                lambda: ops.small_tn(rand(4, 8), rand(5, 8)), lambda: ops.small_nt(rand(4, 8).float(), rand(8, 8)),
                lambda: ops.small_nt(rand(8, 4).t(), rand(8, 8)), lambda: ops.small_nt(rand(0, 8), rand(8, 8)),
                lambda: ops.small_nt(rand(65)[1:].view(8, 8), rand(8, 8)), lambda: ops.small_nt(rand(8, 8).cpu(), rand(8, 8))):
        with pytest.raises(RuntimeError):
            bad()
    for rows in (1, 64, 300, 5000):
        for cols in (8, 512, 4096):
            for total in (8, 128, 1000, 8000):
                edge, parts = ops.small_cut(rows, cols, total)
                assert edge in (64, 128) and (parts == 1 or total >= 128 * parts)
    assert ops.small_cut(256, 256, 256) == (64, 1) and ops.small_cut(512, 512, 8000)[1] > 1
    assert ops.small_cut(4096, 4096, 256) == (128, 1)


def _grads(y, inputs, g):
    return torch.autograd.grad(y, inputs, g, retain_graph=True)


@gpu
@cuda
@pytest.mark.parametrize("T,N,K", [(256, 512, 256), (100, 1024, 2048), (700, 2048, 3584)])
@pytest.mark.parametrize("train_x,train_w", [(True, True), (True, False), (False, True)])
def test_layer(T, N, K, train_x, train_w):
    torch.manual_seed(0)
    lin = nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16).requires_grad_(train_w)
    x, g = rand(2, T // 2, K).requires_grad_(train_x), rand(2, T // 2, N)
    y = L.linear(lin, x)
    assert "SmallLinear" in y.grad_fn.name()
    close(y, x.double() @ lin.weight.double().t(), K)
    inputs = [t for t in (x, lin.weight) if t.requires_grad]
    got = dict(zip(map(id, inputs), _grads(y, inputs, g)))
    flat = g.flatten(0, 1).double()
    if train_x:
        close(got[id(x)], g.double() @ lin.weight.double(), N)
        (alone,) = _grads(y, [x], g)
        assert torch.equal(alone, got[id(x)])
    if train_w:
        close(got[id(lin.weight)], flat.t() @ x.flatten(0, 1).double(), T)
    for strange in (g.transpose(0, 1).contiguous().transpose(0, 1), g[..., :1].expand(g.shape)):
        for a, b in zip(_grads(y, inputs, strange), _grads(y, inputs, strange.contiguous())):
            assert torch.equal(a, b)
    with torch.no_grad():
        assert L.linear(lin, x).grad_fn is None


@gpu
@cuda
def test_gradients_that_are_recorded_or_batched():
    torch.manual_seed(0)
    lin = nn.Linear(64, 128, bias=False, device="cuda", dtype=torch.bfloat16)
    x, g = rand(32, 64).requires_grad_(), rand(3, 32, 128)
    inputs, twice = (x, lin.weight), []
    for y in (L.linear(lin, x), F.linear(x, lin.weight)):
        first = torch.autograd.grad(y, inputs, g[0], create_graph=True)
        twice.append(torch.autograd.grad(sum((t.float() ** 2).sum() for t in first), inputs))
    for a, b in zip(*twice):
        assert torch.equal(a, b)
    batched = torch.autograd.grad(L.linear(lin, x), inputs, g, is_grads_batched=True)
    for i in range(3):
        close(batched[0][i], g[i].double() @ lin.weight.double(), 128)
        close(batched[1][i], g[i].double().t() @ x.double(), 32)


@gpu
@cuda
def test_what_stays_the_module():
    T, N, K = 64, 128, 256
    x = rand(T, K).requires_grad_()

    def own(lin, x=x):
        return "SmallLinear" in L.linear(lin, x).grad_fn.name()

    def make(n=N, k=K, **kw):
        return nn.Linear(k, n, device="cuda", dtype=torch.bfloat16, **{"bias": False, **kw})

    assert own(make()) and not own(make(bias=True)) and not own(make(n=100)) and not own(make(k=252), x[:, :252])
    assert own(make(), rand(2 * T, K).requires_grad_()[::2])       # strides of its own: the library's, in the same node
    for hook in ("register_forward_hook", "register_full_backward_hook"):
        lin, seen = make(), []
        handle = getattr(lin, hook)(lambda *a: seen.append(1) and None)
        L.linear(lin, x).sum().backward()
        assert seen == [1]
        handle.remove()
        assert own(lin)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not own(make())
    from torch.utils.flop_counter import FlopCounterMode

    with FlopCounterMode(display=False) as count:
        L.linear(make(), x).sum().backward()
    assert count.get_total_flops() == 6 * T * N * K
    lin = make()
    out = torch.func.vmap(lambda t: L.linear(lin, t))(x.detach().view(4, -1, K).requires_grad_())
    assert out.shape == (4, T // 4, N)


@gpu
@cuda
def test_a_mode_around_the_backward_alone():
    """It sees the products, as it does those of the module's own call."""
    from torch.utils.flop_counter import FlopCounterMode

    T, N, K = 64, 128, 256
    torch.manual_seed(0)
    lin = nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16)
    x, g = rand(T, K).requires_grad_(), rand(T, N)
    y = L.linear(lin, x)
    assert "SmallLinear" in y.grad_fn.name()
    with FlopCounterMode(display=False) as count:
        dx, dw = _grads(y, (x, lin.weight), g)
    assert count.get_total_flops() == 4 * T * N * K
    close(dx, g.double() @ lin.weight.double(), N)
    close(dw, g.double().t() @ x.double(), T)
    with torch.autograd.forward_ad.dual_level(), FlopCounterMode(display=False) as count:
        _grads(y, (lin.weight,), g)
    assert count.get_total_flops() == 2 * T * N * K


@gpu
@cuda
@pytest.mark.parametrize("kept", ["hooks", "cpu", "checkpoint", "reentrant"])
def test_what_is_kept_for_the_backward(kept):
    from torch.utils.checkpoint import checkpoint

    lin = nn.Linear(256, 128, bias=False, device="cuda", dtype=torch.bfloat16)
    x, g, seen = rand(64, 256).requires_grad_(), rand(64, 128), []
    if kept == "hooks":
        with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t, lambda t: t):
            y = L.linear(lin, x)
        assert sorted(seen) == sorted([x.shape, lin.weight.shape])
    elif kept == "cpu":
        with torch.autograd.graph.save_on_cpu():
            y = L.linear(lin, x)
    else:
        y = checkpoint(lambda t: L.linear(lin, t), x, use_reentrant=kept == "reentrant")
    (y * g).sum().backward()
    close(x.grad, g.double() @ lin.weight.double(), 128)
    close(lin.weight.grad, g.double().t() @ x.double(), 64)
    z = L.linear(lin, x)
    with torch.no_grad():
        lin.weight.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        z.sum().backward()


def test_sizes():
    assert L.small(1, 8, 8) and L.small(1000, 2048, 2048) and not L.small(1024, 2048, 2048)
    assert L.small(2000, 2048, 2048, L.MAX_SMALL_DW) and not L.small(0, 8, 8)
    assert not L.small(4, 12, 8) and not L.small(4, 8, 12) and not L.small(1 << 23, 8, 8)
