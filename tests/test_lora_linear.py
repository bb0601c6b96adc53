"""An adapted layer's product with the adapter's behind its sums (csrc/linear_grad.hip: lora_linear)."""

import pytest
import torch

from automodel_amd.ops import _backend
from automodel_amd.peft import lora

gpu = pytest.mark.gpu
cuda = pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")


def rand(*shape, std=1.0):
    return (torch.randn(*shape, device="cuda") * std).bfloat16()


# one row, every height of a tile, columns that end within one, sums in parts; ranks filled up with zeros to 32 and 64
@gpu
@cuda
@pytest.mark.parametrize("T,N,K,r,scale", [
    (1, 64, 128, 32, 2.0), (127, 320, 128, 8, 0.5), (200, 64, 192, 40, 1.0), (300, 576, 8256, 64, 2.0), (513, 4096, 1024, 16, 4.0),
    (1025, 2816, 512, 32, 0.3), (3003, 1088, 256, 48, 2.0), (4100, 4160, 128, 24, 1.0),
])
def test_sum(T, N, K, r, scale):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(T)
    x, w, a, b = rand(T, K), rand(N, K, std=K ** -0.5), rand(r, K, std=K ** -0.5), rand(N, r, std=0.3)
    y, t = hip_ops().lora_linear(x, w, a, b, scale)
    before, turned = hip_ops().lora_forward(x @ w.t(), x, a, b, scale)
    assert torch.equal(t, turned)
    s = (scale * (x.double() @ a.double().t())).bfloat16().double()      # as the kernel rounds it
    own = x.double() @ w.double().t() + s @ b.double().t()
    # one rounding to 8 bits; a sum in 24 bits may round another way
    assert (y.double() - own).norm() <= 2.0 ** -9 * 1.05 * own.norm()
    ref = x.double() @ w.double().t() + scale * (x.double() @ a.double().t()) @ b.double().t()
    # and no further off than the product rounded before the sum (t rounded behind the scale: by chance more or less)
    assert (y.double() - ref).norm() <= 1.02 * (before.double() - ref).norm()


@gpu
@cuda
@pytest.mark.parametrize("r", [8, 32, 40])
def test_infinite_rows_and_edges(r):
    """An infinite row stays one, and nothing beyond the operands is read into a result."""
    from automodel_amd.ops._backend import hip_ops

    def within(v):
        whole = torch.full((v.numel() + 65536,), float("inf"), device="cuda", dtype=torch.bfloat16)
        whole[: v.numel()] = v.flatten()
        return whole[: v.numel()].view(v.shape)
    torch.manual_seed(0)
    x, w, a, b = (within(torch.rand(s) + 0.1) for s in ((70, 192), (64, 192), (r, 192), (64, r)))
    x[3, 100], x[5, 1] = float("inf"), -float("inf")
    y, t = hip_ops().lora_linear(x, w, a, b, 2.0)
    assert (y[3] == float("inf")).all() and (y[5] == -float("inf")).all() and y.isfinite().all(1).sum() == 68
    assert (t[r:] == 0).all() and (t[:, 70:] == 0).all()


@gpu
@cuda
def test_refusals():
    from automodel_amd.ops._backend import hip_ops

    op, good = hip_ops().lora_linear, (rand(8, 128), rand(64, 128), rand(32, 128), rand(64, 32))
    op(*good, 1.0)
    for at, bad in ((0, rand(8, 192)), (0, rand(0, 128)), (0, rand(128, 8).t()), (0, rand(1025)[1:].view(8, 128)),
                    (0, rand(8, 128).float()), (1, rand(72, 128)), (2, rand(12, 128)), (2, rand(72, 128)), (3, rand(64, 40)),
                    (3, rand(128, 32)), (3, rand(64, 32).cpu())):
        with pytest.raises(RuntimeError):
            op(*good[:at], bad, *good[at + 1:], 1.0)


class Kernels:
    """The kernels by their definitions, for the function around them."""

    used = 0

    def lora_linear(self, x, w, a, b, scale):
        Kernels.used += 1
        t = x @ a.t()
        return x @ w.t() + scale * t @ b.t(), torch.nn.functional.pad(t.t(), (0, -x.shape[0] % 64, 0, -a.shape[0] % 32))

    def lora_grads(self, g, x, a, b, tt, scale):
        dt, fill = scale * g @ b, (0, -a.shape[0] % 32)
        pad = torch.nn.functional.pad
        return dt.t() @ x, scale * g.t() @ tt[:a.shape[0], :x.shape[0]].t(), pad(dt, fill), pad(a.t(), fill)

    def linear_dx_extra(self, g, w, t, a_t):
        return g @ w + t @ a_t.t()


@pytest.mark.parametrize("rank", [8, 32, 40])
def test_function(monkeypatch, rank):
    monkeypatch.setattr(_backend, "hip_ops", Kernels)
    monkeypatch.setattr(lora, "_plain", lambda *ts: True)
    Kernels.used = 0
    torch.manual_seed(rank)
    x, w, a, b = (torch.randn(s, dtype=torch.float64) for s in ((10, 192), (64, 192), (rank, 192), (64, rank)))
    g, wrt = torch.randn(10, 64, dtype=torch.float64), [v.requires_grad_() for v in (x, a, b)]
    own = lora._LoRALinear.apply(x, w, a, b, 0.5)
    ref = x @ w.t() + 0.5 * (x @ a.t()) @ b.t()
    torch.testing.assert_close(own, ref)
    assert Kernels.used == 1
    for twice in (False, True):
        got, want = (torch.autograd.grad(v, wrt, g, create_graph=twice, retain_graph=True) for v in (own, ref))
        torch.testing.assert_close(got, want)
        if twice:
            got, want = (torch.autograd.grad(sum((v * v).sum() for v in vs), wrt) for vs in (got, want))
            torch.testing.assert_close(got, want)


def test_which_layers_are_one_product():
    assert lora.adapted_own(8192, 28672, 4096) and lora.adapted_own(408, 6144, 4096) and lora.adapted_own(1000, 2048, 1024)
    # few rows; few tiles; a weight's reads; half of the chip
    for sizes in ((96, 6144, 4096), (168, 2048, 2048), (200, 1024, 4096), (128, 28672, 4096), (384, 10240, 2560)):
        assert not lora.adapted_own(*sizes)
    for sizes in ((1 << 23, 64, 128), (8192, 4096, 64)):                   # the kernel refuses these
        assert not lora.adapted_own(*sizes)


class Two(Kernels):
    """Those of a layer whose product and adapter are two."""

    def lora_linear(self, *_):
        raise AssertionError

    def lora_forward(self, y, x, a, b, scale):
        t = x @ a.t()
        return y + scale * t @ b.t(), torch.nn.functional.pad(t.t(), (0, -x.shape[0] % 64, 0, -a.shape[0] % 32))


def test_two_products(monkeypatch):
    monkeypatch.setattr(_backend, "hip_ops", Two)
    monkeypatch.setattr(lora, "_plain", lambda *ts: True)
    torch.manual_seed(0)
    x, w, a, b = (torch.randn(s, dtype=torch.float64) for s in ((10, 192), (64, 192), (8, 192), (64, 8)))
    g, wrt = torch.randn(10, 64, dtype=torch.float64), [v.requires_grad_() for v in (x, a, b)]
    own = lora._LoRALinear.apply(x, w, a, b, 0.5, False)
    ref = x @ w.t() + 0.5 * (x @ a.t()) @ b.t()
    torch.testing.assert_close(own, ref)
    torch.testing.assert_close(torch.autograd.grad(own, wrt, g), torch.autograd.grad(ref, wrt, g))
