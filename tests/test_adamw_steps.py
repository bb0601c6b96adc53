"""AdamW over many tensors at once: chunk edges, mixed steps, more tensors than one launch takes."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


def reference(x, t, lr, b1, b2, eps, wd):
    p, g, master, m, v = (y.double() for y in x)
    m = b1 * m + (1 - b1) * g
    v = b2 * v + (1 - b2) * g * g
    w = master * (1 - lr * wd)
    return w - lr / (1 - b1 ** t) * m / ((v / (1 - b2 ** t)).sqrt() + eps), m, v


@pytest.mark.parametrize("sizes", [
    [4], [4096, 4100, 4092, 8, 16384], [64 + 4 * i for i in range(95)], [23_000_000, 12, 4096],
])
def test_against_f64(sizes):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    hyper = (1e-2, 0.9, 0.95, 1e-8, 0.1)
    steps = [1 + i % 3 for i in range(len(sizes))]
    xs = []
    for n in sizes:
        w = torch.randn(n, device="cuda")
        xs.append([w.bfloat16(), torch.randn(n, device="cuda").bfloat16(), w,
                   0.1 * torch.randn(n, device="cuda"), 0.1 * torch.rand(n, device="cuda")])
    want = [reference(x, t, *hyper) for x, t in zip(xs, steps)]
    hip_ops().adamw_steps(*[list(c) for c in zip(*xs)], steps, *hyper)
    for (p, _, w, m, v), (rw, rm, rv) in zip(xs, want):
        # a dozen float32 operations (2^-24 each) on values of up to a few units
        for got, ref in ((w, rw), (m, rm), (v, rv)):
            assert ((got.double() - ref).abs() <= 12 * 2.0 ** -24 * (1 + ref.abs())).all()
        assert torch.equal(p, w.bfloat16())
