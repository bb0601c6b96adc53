"""Gradients of an adapted layer's autograd functions, with the kernels' part played by Python in 64 bits."""

import pytest
import torch
import torch.nn.functional as F

from automodel_amd.ops import _backend
from automodel_amd.peft import lora


class Kernels:
    """csrc/lora.hip and lora_grad.hip by their definitions."""

    calls = 0

    @staticmethod
    def _filled(r):
        return 32 if r <= 32 else 64

    def lora_apply(self, y, x, A, B, scale):
        Kernels.turned = False
        t = x @ A.t()
        return y + scale * t @ B.t(), F.pad(t, (0, self._filled(A.shape[0]) - A.shape[0]))

    def lora_forward(self, y, x, A, B, scale):
        out, t = self.lora_apply(y, x, A, B, scale)
        Kernels.turned = True
        return out, F.pad(t.t(), (0, -x.shape[0] % 64))

    def lora_grads(self, g, x, A, B, tt, scale):
        Kernels.calls += 1
        M, r = x.shape[0], A.shape[0]
        assert M > 0
        dt = scale * g @ B
        fill = (0, self._filled(r) - r)
        return dt.t() @ x, scale * g.t() @ tt[:r, :M].t(), F.pad(dt, fill), F.pad(A.t(), fill)

    def linear_dx_extra(self, g, w, t, a_t):
        return g @ w + t @ a_t.t()


@pytest.fixture
def kernels(monkeypatch):
    monkeypatch.setattr(_backend, "hip_ops", Kernels)
    monkeypatch.setattr(lora, "_plain", lambda *ts: True)
    Kernels.calls = 0
    return Kernels


def layer(M, rank, H=24, O=40):
    torch.manual_seed(rank)
    shapes = (M, H), (O, H), (rank, H), (O, rank)
    x, w, a, b = (torch.randn(s, dtype=torch.float64) for s in shapes)
    return x.requires_grad_(), w, a.requires_grad_(), b.requires_grad_(), torch.randn(M, O, dtype=torch.float64)


def kinds(x, w, a, b):
    """The layer by either function, and by torch's operations."""
    return {"linear": lambda: lora._LoRALinear.apply(x, w, a, b, 0.5),
            "fused": lambda: lora._FusedLoRAFn.apply(F.linear(x, w), x, a, b, 0.5),
            "torch": lambda: F.linear(x, w) + 0.5 * F.linear(F.linear(x, a), b)}


@pytest.mark.parametrize("rank", [8, 32, 40])
@pytest.mark.parametrize("kind", ["linear", "fused"])
def test_once_and_twice(kernels, kind, rank):
    x, w, a, b, g = layer(10, rank)
    make = kinds(x, w, a, b)
    got, want = (torch.autograd.grad(make[k](), (x, a, b), g) for k in (kind, "torch"))
    assert kernels.calls == 1
    for u, v in zip(got, want):
        torch.testing.assert_close(u, v)
    # every first gradient's part in the second ones
    for i in range(3):
        second = []
        for k in (kind, "torch"):
            gg = g.clone().requires_grad_()
            first = torch.autograd.grad(make[k](), (x, a, b), gg, create_graph=True)
            second.append(torch.autograd.grad(first[i].square().sum(), (x, a, b, gg), allow_unused=True,
                                              materialize_grads=True))
        for u, v in zip(*second):
            torch.testing.assert_close(u, v)


@pytest.mark.parametrize("rank", [8, 32])
@pytest.mark.parametrize("kind", ["linear", "fused"])
def test_no_rows(kernels, kind, rank):
    x, w, a, b, g = layer(0, rank)
    for d, of in zip(torch.autograd.grad(kinds(x, w, a, b)[kind](), (x, a, b), g), (x, a, b)):
        assert d.shape == of.shape and not d.any()


@pytest.mark.parametrize("rank", [8, 40])
def test_a_weight_that_came_back_in_another_form(kernels, monkeypatch, rank):
    x, w, a, b, g = layer(10, rank)
    make = kinds(x, w, a, b)
    monkeypatch.setattr(lora, "_plain", lambda *ts: all(t.data_ptr() != w.data_ptr() for t in ts))
    got, want = (torch.autograd.grad(make[k](), (x, a, b), g) for k in ("linear", "torch"))
    assert kernels.calls == 1
    for u, v in zip(got, want):
        torch.testing.assert_close(u, v)


@pytest.mark.parametrize("rank", [8, 32])
def test_what_is_kept(kernels, rank):
    """t^T only for a backward by the kernels; a followed forward keeps t for torch's products."""
    x, w, a, b, g = layer(10, rank)
    y = F.linear(x, w).detach()
    run = lambda: lora._FusedLoRAFn.apply(y, x, a, b, 0.5, torch.is_grad_enabled())
    with torch.no_grad():
        out = run()
        assert not kernels.turned
    assert torch.equal(run(), out) and kernels.turned
    from torch.utils.flop_counter import FlopCounterMode

    make = kinds(x, w, a, b)
    with FlopCounterMode(display=False):
        z = make["fused"]()
    assert not kernels.turned
    got, want = (torch.autograd.grad(v, (x, a, b), g) for v in (z, make["torch"]()))
    assert kernels.calls == 0
    for u, v in zip(got, want):
        torch.testing.assert_close(u, v)


@pytest.mark.parametrize("rank", [8, 32])
@pytest.mark.parametrize("kind", ["linear", "fused"])
def test_batched(kernels, kind, rank):
    x, w, a, b, g = layer(10, rank)
    make, gs = kinds(x, w, a, b), torch.stack([g, g.flip(0)])
    got, want = (torch.autograd.grad(make[k](), (x, a, b), gs, is_grads_batched=True) for k in (kind, "torch"))
    assert kernels.calls == 0
    for u, v in zip(got, want):
        torch.testing.assert_close(u, v)
