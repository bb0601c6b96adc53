"""Linear layers of decode steps: tiles, tails and epilogues of both kernels."""

import pytest
import torch
import torch.nn as nn

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]

# a bf16 output (8 bits) is off by 2^-8 of itself at most; float32 sums of K products of
# either sign by far less than 1e-4 of the largest
HALF_UNIT = 2.0 ** -8


def check(y, ref):
    rounding = HALF_UNIT if y.dtype == torch.bfloat16 else 0
    err = (y.double() - ref).abs()
    assert (err <= rounding * ref.abs() + 1e-4 * ref.abs().max()).all()


@pytest.mark.parametrize("B", [1, 2, 3, 4, 8, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("K,ns", [
    (8, [1]), (520, [16, 17, 3]), (2048, [300]), (4104, [64, 1, 15]), (6656, [40]), (136, [8192, 70]),
])
@pytest.mark.parametrize("glu", [False, True])
def test_several_weights(B, K, ns, glu):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    x = torch.randn(B, K, device="cuda").bfloat16()
    ns = [ns[0]] * 2 if glu else ns
    ws = [torch.randn(n, K, device="cuda").bfloat16() * K ** -0.5 for n in ns]
    ys = hip_ops().decode_rows(x, ws, glu)
    refs = [x.double() @ w.double().t() for w in ws]
    if glu:
        refs = [nn.functional.silu(refs[0]) * refs[1]]
    assert len(ys) == len(refs)
    for y, ref in zip(ys, refs):
        check(y, ref)


# every split of the rows of W: 16, 32 and 64 a workgroup, alone on a CU or not, the last ones partly empty
@pytest.mark.parametrize("N", [4090, 5110, 6150, 9210, 10250, 15370, 21510, 32010])
@pytest.mark.parametrize("B,K", [(1, 2056), (2, 2056), (2, 4096), (2, 5000), (8, 264), (8, 520), (16, 2056),
                                 (32, 520), (32, 264), (32, 4104), (64, 520), (33, 4104)])
def test_every_split_of_the_rows(N, B, K):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    x = torch.randn(B, K, device="cuda").bfloat16()
    w = torch.randn(N, K, device="cuda").bfloat16() * K ** -0.5
    check(hip_ops().decode_rows(x, [w])[0], x.double() @ w.double().t())


@pytest.mark.parametrize("T", [1, 2, 3, 5, 20, 40])
@pytest.mark.parametrize("K,sizes", [(512, [64, 64, 64]), (2056, [48, 48, 16]), (264, [4096, 4096, 64])])
def test_groups_and_epilogues(T, K, sizes):
    from automodel_amd.ops._backend import hip_ops
    from automodel_amd.serving.decode_linear import project, project_grouped

    torch.manual_seed(0)
    lin = nn.Linear(K, sum(sizes), bias=False, device="cuda", dtype=torch.bfloat16)
    xs = torch.randn(len(sizes), T, K, device="cuda").bfloat16()
    with torch.no_grad():
        ys = project_grouped(lin, xs, sizes)
        y = project(lin, xs[0], relu2=True, out_f32=True)
    for y_, x, w in zip(ys, xs, lin.weight.split(sizes)):
        check(y_, x.double() @ w.double().t())
    assert y.dtype == torch.float32
    check(y, (xs[0].double() @ lin.weight.double().t()).clamp(min=0) ** 2)


def test_refused_and_general_path():
    """What the kernels don't take goes through the layers themselves."""
    from automodel_amd.serving.decode_linear import decode_rows

    lin = nn.Linear(64, 32, bias=False, device="cuda", dtype=torch.bfloat16)
    biased = nn.Linear(64, 32, device="cuda", dtype=torch.bfloat16)
    hooked = nn.Linear(64, 32, bias=False, device="cuda", dtype=torch.bfloat16)
    hooked.register_forward_hook(lambda *a: None)
    x = torch.randn(2, 1, 64, device="cuda").bfloat16()
    assert decode_rows([lin], x) is None                        # autograd
    with torch.no_grad():
        (y,) = decode_rows([lin], x)
        assert y.shape == (2, 1, 32)
        torch.testing.assert_close(y, lin(x))
        for lins, rows in (([biased], x), ([hooked], x), ([lin], x.float()), ([lin], x.expand(2, 17, 64)),
                           ([lin], x[:0]), ([lin], torch.randn(2, 128, device="cuda").bfloat16()[:, ::2]),
                           ([lin], torch.randn(129, device="cuda").bfloat16()[1:].view(2, 64)),
                           ([lin.float()], x)):
            assert decode_rows(lins, rows) is None
