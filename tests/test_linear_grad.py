"""Gradients of linear layers on 256 x 256 tiles: edges of the tiles and of the summed index, and
which calls of a layer come to them."""

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from automodel_amd.ops import linear as L

gpu = pytest.mark.gpu
cuda = pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")


def close(got, want):
    # f32 sums, rounded to bf16 once: 8 bits, so half a unit is at most 2^-8 of a value (results of 64
    # elements come to 0.54 of that, large ones to 0.42). The f32 sums of up to 4096 products are
    # off by 1e-6 of the result's size, which 2% of it covers
    assert got.shape == want.shape
    assert (got.double() - want).norm() <= 2.0 ** -8 * 1.02 * want.norm()


def rand(*shape):
    return torch.randn(*shape, device="cuda").bfloat16()


@gpu
@cuda
@pytest.mark.parametrize("T", [1, 7, 31, 32, 33, 63, 64, 65, 95, 97, 130, 1001])
@pytest.mark.parametrize("N,K", [(8, 8), (256, 512), (264, 248), (1000, 136)])
def test_weight_gradient(T, N, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)
    g, x = rand(T, N), rand(T, K)
    close(hip_ops().linear_dw(g, x), g.double().t() @ x.double())


@gpu
@cuda
@pytest.mark.parametrize("T", [1, 8, 255, 256, 257, 1001])
@pytest.mark.parametrize("N,K", [(64, 8), (128, 512), (192, 248), (320, 1000), (1024, 136)])
def test_input_gradient(T, N, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)
    g, w = rand(T, N), rand(N, K)
    close(hip_ops().linear_dx(g, w), g.double() @ w.double())


# tiles of 128 to 256 rows, sums in parts of which the last is shorter
@gpu
@cuda
@pytest.mark.parametrize("T,N,K", [
    (512, 264, 248), (513, 1000, 136), (640, 520, 1032), (1023, 264, 8), (1025, 8, 520), (1100, 2048, 1032),
    (2050, 136, 2056), (4100, 1032, 1032), (700, 4104, 4096), (300, 6152, 2568), (260, 5000, 7688),
])
def test_weight_gradient_of_cut_tiles(T, N, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)
    g, x = rand(T, N), rand(T, K)
    close(hip_ops().linear_dw(g, x), g.double().t() @ x.double())


@gpu
@cuda
@pytest.mark.parametrize("T,N,K", [
    (1, 1024, 136), (129, 576, 8), (257, 1088, 520), (300, 2048, 248), (1001, 1024, 1032), (500, 6144, 1536),
    (1001, 2816, 2048), (1300, 512, 5000), (2050, 640, 4104), (161, 704, 8),
])
def test_input_gradient_of_cut_tiles(T, N, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)
    g, w = rand(T, N), rand(N, K)
    close(hip_ops().linear_dx(g, w), g.double() @ w.double())


@gpu
@cuda
def test_how_sums_and_tiles_are_cut():
    from automodel_amd.ops._backend import hip_ops

    cut = hip_ops().linear_grad_cut
    assert cut(True, 8192, 4096, 4096) == [256, 1] and cut(False, 8192, 4096, 4096) == [256, 1]
    assert cut(True, 8192, 6144, 4096) == [192, 1] and cut(True, 8192, 2048, 2048) == [128, 2]
    assert cut(False, 1001, 6144, 1536) == [128, 4] and cut(False, 300, 64, 8) == [128, 1]
    for dw in (True, False):
        for T in (1, 63, 256, 500, 1001, 4096, 8192):
            for N in (64, 128, 320, 1024, 2816, 14336):
                for K in (8, 520, 2048, 4096):
                    height, parts = cut(dw, T, N, K)
                    total = T if dw else N
                    per = -(-total // (64 * parts)) * 64
                    assert height in (128, 160, 192, 224, 256)
                    assert parts == 1 or (per >= 256 and total - (parts - 1) * per >= 128)


@gpu
@cuda
@pytest.mark.parametrize("T,N,K", [(6001, 2048, 2048), (3003, 2816, 2048), (4096, 1024, 2048)])
def test_layer_of_cut_tiles(T, N, K):
    torch.manual_seed(0)
    lin = nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16)
    x, g = rand(T, K).requires_grad_(), rand(T, N)
    assert L.weight_grad_cut(T, N, K) and L.input_grad_cut(T, N, K)
    y = L.linear(lin, x)
    assert "_Linear" in type(y.grad_fn).__name__ and torch.equal(y, lin(x))
    dx, dw = torch.autograd.grad(y, (x, lin.weight), g)
    close(dx, g.double() @ lin.weight.double())
    close(dw, g.double().t() @ x.double())


@gpu
@cuda
def test_refusals():
    from automodel_amd.ops._backend import hip_ops

    ops = hip_ops()
    for bad in (lambda: ops.linear_dw(rand(4, 12), rand(4, 8)), lambda: ops.linear_dw(rand(4, 8), rand(5, 8)),
                lambda: ops.linear_dw(rand(4, 8).float(), rand(4, 8)), lambda: ops.linear_dw(rand(8, 4).t(), rand(4, 8)),
                lambda: ops.linear_dx(rand(4, 32), rand(32, 8)), lambda: ops.linear_dx(rand(4, 64), rand(64, 12)),
                lambda: ops.linear_dx(rand(4, 64), rand(64, 8).cpu())):
        with pytest.raises(RuntimeError):
            bad()


@gpu
@cuda
@pytest.mark.parametrize("T,N,K,dw,dx", [
    (1040, 4096, 4096, True, False), (4095, 1088, 4096, False, True), (2048, 4096, 4096, True, False),
    (4096, 4096, 4096, True, True), (1000, 4096, 4096, False, False), (4096, 4100, 4096, False, False),
    (300, 4096, 4096, False, False), (16384, 192, 4096, False, False), (200, 8192, 8192, False, False),
])
@pytest.mark.parametrize("train_x,train_w", [(True, True), (True, False), (False, True)])
def test_layer(monkeypatch, T, N, K, dw, dx, train_x, train_w):
    torch.manual_seed(0)
    lin = nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16).requires_grad_(train_w)
    x = rand(1, T, K).requires_grad_(train_x)
    g = rand(1, T, N)
    assert L.weight_grad_wins(T, N, K) == dw and L.input_grad_wins(T, N, K) == dx
    y = L.linear(lin, x)
    # whole tiles, or cut ones of sizes from 256 on and 2^33 products
    cut = min(T, N, K) >= 256 and T * N * K >= 1 << 33 and N % 64 == 0
    own = (dw or cut) and train_w or (dx or cut) and train_x
    assert ("_Linear" in type(y.grad_fn).__name__) == own
    assert torch.equal(y, lin(x))
    inputs = [t for t in (x, lin.weight) if t.requires_grad]
    got = dict(zip(map(id, inputs), torch.autograd.grad(y, inputs, g, retain_graph=True)))
    if train_x:
        close(got[id(x)][0], g[0].double() @ lin.weight.double())
    if train_w:
        close(got[id(lin.weight)], g[0].double().t() @ x[0].double())
    if own and train_x and train_w:       # gradients of gradients, as F.linear has them
        twice = []
        for z in (y, F.linear(x, lin.weight)):
            first = torch.autograd.grad(z, inputs, g, create_graph=True)
            twice.append(torch.autograd.grad(sum((t.float() ** 2).sum() for t in first), inputs))
        for a, b in zip(*twice):
            assert torch.equal(a, b)


@gpu
@cuda
@pytest.mark.parametrize("T,N,K", [(4096, 4096, 4096), (2000, 2816, 2048)])        # whole tiles, and cut ones
def test_calls_that_stay_the_module(monkeypatch, T, N, K):
    x = rand(T, K).requires_grad_()

    def own(lin, x=x):
        return "_Linear" in type(L.linear(lin, x).grad_fn).__name__

    def make(**kw):
        return nn.Linear(K, N, device="cuda", dtype=torch.bfloat16, **{"bias": False, **kw})

    assert own(make())
    assert not own(make(bias=True))
    assert own(make(), x.view(2, -1, K)) and not own(make(), x[:100])
    for hook in ("register_forward_hook", "register_forward_pre_hook", "register_full_backward_hook",
                 "register_full_backward_pre_hook"):
        lin, seen = make(), []
        handle = getattr(lin, hook)(lambda *a: seen.append(1) and None)
        L.linear(lin, x).sum().backward()
        assert seen == [1]
        handle.remove()
        assert own(lin)

    class Other(nn.Linear):
        pass

    assert not own(Other(K, N, bias=False, device="cuda", dtype=torch.bfloat16))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not own(make())
    with torch.no_grad():
        assert L.linear(make(), x).grad_fn is None
    from torch.utils.flop_counter import FlopCounterMode

    lin = make()
    with FlopCounterMode(display=False) as count:
        L.linear(lin, x).sum().backward()
    assert count.get_total_flops() == 6 * T * N * K
    import torch.autograd.forward_ad as fwd

    with fwd.dual_level():
        y = L.linear(lin, fwd.make_dual(x.detach().requires_grad_(), torch.ones_like(x)))
        close(fwd.unpack_dual(y).tangent, torch.ones_like(x).double() @ lin.weight.double().t())
    out = torch.func.vmap(lambda t: L.linear(lin, t))(x.detach().view(4, -1, K).requires_grad_())
    assert out.shape == (4, T // 4, N)


@gpu
@cuda
@pytest.mark.parametrize("rows", [4096, 1000])
def test_without_the_kernels(monkeypatch, rows):
    lin = nn.Linear(4096, 4096, bias=False, device="cuda", dtype=torch.bfloat16)
    x = rand(rows, 4096).requires_grad_()
    assert "_Linear" in type(L.linear(lin, x).grad_fn).__name__
    monkeypatch.setattr(L, "_built", lambda: False)
    assert "_Linear" not in type(L.linear(lin, x).grad_fn).__name__


class _Halved(torch.overrides.TorchFunctionMode):
    """Linears with half the weight, as a mode for rounded weights would put them in place."""

    def __torch_function__(self, func, types, args=(), kwargs=None):
        if func is F.linear:
            args = (args[0], args[1] * 0.5)
        return func(*args, **(kwargs or {}))


def test_function_modes():
    lin = nn.Linear(16, 8, bias=False)
    assert L._unseen(lin)
    with torch.device("cpu"):
        assert L._unseen(lin)
        with _Halved():
            assert not L._unseen(lin)
    assert L._unseen(lin)


@gpu
@cuda
def test_a_mode_in_the_place_of_linears():
    lin = nn.Linear(4096, 4096, bias=False, device="cuda", dtype=torch.bfloat16)
    x, g = rand(4096, 4096).requires_grad_(), rand(4096, 4096)
    with _Halved():
        y = L.linear(lin, x)
    dx, dw = torch.autograd.grad(y, (x, lin.weight), g)
    close(dx, g.double() @ lin.weight.double() * 0.5)
    close(dw, g.double().t() @ x.double() * 0.5)
    with torch.device("cuda"):
        assert "_Linear" in type(L.linear(lin, x).grad_fn).__name__


def test_what_is_built(monkeypatch):
    inference = type("Inference", (), {"flash_attn_fwd": None})()
    monkeypatch.setattr(torch.ops, "amd_ops", inference, raising=False)
    for found in (False, True):
        monkeypatch.setattr(L, "ops_available", lambda: found)
        assert not L._built()
    inference.linear_dw = lambda *a: None
    assert L._built()


@gpu
@cuda
def test_backward_that_is_followed():
    from torch.utils.flop_counter import FlopCounterMode

    from automodel_amd.loss.linear_ce import fused_linear_cross_entropy

    T, N, K = 4096, 4096, 4096
    torch.manual_seed(0)
    lin = nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16)
    x, g = rand(T, K).requires_grad_(), rand(2, T, N)
    y = L.linear(lin, x)
    assert "_Linear" in type(y.grad_fn).__name__
    with FlopCounterMode(display=False) as count:       # around the backward alone
        torch.autograd.grad(y, (x, lin.weight), g[0], retain_graph=True)
    assert count.get_total_flops() == 4 * T * N * K
    dx, dw = torch.autograd.grad(y, (x, lin.weight), g, is_grads_batched=True)
    for i in range(2):
        close(dx[i], g[i].double() @ lin.weight.double())
        close(dw[i], g[i].double().t() @ x.double())
    # the head: logits are kept, so that its backward has two products
    h, labels = rand(T, 2048).requires_grad_(), torch.randint(16384, (T,), device="cuda")
    head = rand(16384, 2048).requires_grad_()
    loss = fused_linear_cross_entropy(h, head, labels)
    with FlopCounterMode(display=False) as count:
        loss.backward()
    assert count.get_total_flops() == 4 * T * 16384 * 2048


@gpu
@cuda
@pytest.mark.parametrize("kept", ["hooks", "cpu", "checkpoint", "reentrant"])
def test_what_is_kept_for_the_backward(kept):
    from torch.utils.checkpoint import checkpoint

    T, N, K = 4096, 4096, 4096
    torch.manual_seed(0)
    lin = nn.Linear(K, N, bias=False, device="cuda", dtype=torch.bfloat16)
    x, g, seen = rand(T, K).requires_grad_(), rand(T, N), []
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
    close(x.grad, g.double() @ lin.weight.double())
    close(lin.weight.grad, g.double().t() @ x.double())
    z = L.linear(lin, x)
    with torch.no_grad():
        lin.weight.mul_(2)                       # what the backward needs is gone, as with F.linear
    with pytest.raises(RuntimeError, match="modified by an inplace"):
        z.sum().backward()


def test_backward_that_is_followed_elsewhere(monkeypatch):
    # which products a backward takes, with the kernels' part played by Python
    from torch.utils.flop_counter import FlopCounterMode

    class Kernels:
        calls = 0

        def linear_dw(self, g, x):
            Kernels.calls += 1
            return g.t() @ x

        def linear_dx(self, g, w):
            Kernels.calls += 1
            return g @ w

    monkeypatch.setattr(L, "hip_ops", Kernels)
    monkeypatch.setattr(L, "_plain", lambda *ts: all(t.data_ptr() for t in ts))
    for rule in ("weight_grad_wins", "input_grad_wins"):
        monkeypatch.setattr(L, rule, lambda *sizes: True)
    x, w, g = torch.randn(5, 16, requires_grad=True), torch.randn(8, 16, requires_grad=True), torch.randn(2, 5, 8)
    y = L._Linear.apply(x, w)
    one = torch.autograd.grad(y, (x, w), g[0], retain_graph=True)
    assert Kernels.calls == 2
    both = torch.autograd.grad(y, (x, w), g, is_grads_batched=True, retain_graph=True)
    for a, b in zip(one, both):
        torch.testing.assert_close(a, b[0])
    with FlopCounterMode(display=False) as count:
        torch.autograd.grad(y, (x, w), g[0])
    assert Kernels.calls == 2 and count.get_total_flops() == 4 * 5 * 8 * 16


def test_layers_elsewhere():
    lin, seen = nn.Linear(16, 8, bias=False), []
    lin.register_forward_hook(lambda *a: seen.append(1))
    x = torch.randn(3, 16, requires_grad=True)
    assert torch.equal(L.linear(lin, x), F.linear(x, lin.weight)) and seen == [1]
    assert torch.equal(L.weight_grad(x, x), x.t() @ x) and torch.equal(L.input_grad(x, lin.weight.t()), x @ lin.weight.t())


def test_rule():
    # the chip's 256 workgroups per round: whole, three quarters and half rounds
    assert L.weight_grad_wins(8192, 4096, 4096) and L.weight_grad_wins(8192, 6144, 4096)
    assert not L.weight_grad_wins(8192, 2048, 4096) and not L.weight_grad_wins(64, 4096, 4096)
    assert not L.weight_grad_wins(8192, 4100, 4096) and not L.weight_grad_wins(8192, 4096, 4092)
    assert L.input_grad_wins(8192, 6144, 4096) and not L.input_grad_wins(6001, 4096, 4096)
    assert not L.input_grad_wins(8192, 6176, 4096) and not L.input_grad_wins(8192, 4096, 4100)


def test_sizes_beyond_the_kernels_addresses():
    for T, N, K in ((1 << 23, 4096, 4096), (8192, 1 << 23, 4096), (8192, 4096, 1 << 23)):
        assert not L.weight_grad_wins(T, N, K) and not L.input_grad_wins(T, N, K)
    assert L.weight_grad_wins((1 << 23) - 1, 4096, 4096) and L.input_grad_wins(8192, (1 << 23) - 64, 4096)
