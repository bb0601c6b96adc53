"""y + scale * (x A^T) B^T at odd row counts and the smallest widths."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("M,H,O,R", [(1, 64, 64, 32), (33, 128, 320, 32), (200, 4096, 192, 64),
                                     (1000, 192, 4096, 32), (8, 8192, 64, 64), (65, 64, 576, 64)])
@pytest.mark.parametrize("with_y", [True, False])
def test_lora_apply(M, H, O, R, with_y):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    x = torch.randn(M, H, device="cuda").bfloat16()
    A = (torch.randn(R, H, device="cuda") / H ** 0.5).bfloat16()
    B = torch.randn(O, R, device="cuda").bfloat16()
    y = torch.randn(M, O, device="cuda").bfloat16() if with_y else None
    out, t = hip_ops().lora_apply(y, x, A, B, 0.5)
    td = x.double() @ A.double().t()
    # each value is rounded to bf16 once
    assert (t.double() - td).norm() <= 2.0 ** -9 * 1.05 * td.norm()
    ref = 0.5 * (t.double() @ B.double().t()) + (0 if y is None else y.double())
    assert (out.double() - ref).norm() <= 2.0 ** -9 * 1.05 * ref.norm()


@pytest.mark.parametrize("at", [1, 2, 3, 4])
def test_operands_anywhere_in_a_buffer(at):
    from automodel_amd.ops._backend import hip_ops

    def moved(v):
        return torch.cat([v.new_zeros(at), v.flatten()])[at:].view(v.shape)

    torch.manual_seed(0)
    x, A = torch.randn(40, 192, device="cuda").bfloat16(), torch.randn(32, 192, device="cuda").bfloat16()
    B, y = torch.randn(64, 32, device="cuda").bfloat16(), torch.randn(40, 64, device="cuda").bfloat16()
    want = hip_ops().lora_forward(y, x, A, B, 0.5)
    for args in ((y, moved(x), A, B), (y, x, moved(A), B), (y, moved(x), moved(A), B)):
        assert all(torch.equal(a, b) for a, b in zip(hip_ops().lora_forward(*args, 0.5), want))
        assert torch.equal(hip_ops().lora_apply(*args, 0.5)[0], want[0])


def test_more_rows_than_a_grid_is_high():
    from automodel_amd.ops._backend import hip_ops

    M = 65535 * 64 + 33
    torch.manual_seed(0)
    x = torch.randn(M, 64, device="cuda").bfloat16()
    A, B = torch.randn(32, 64, device="cuda").bfloat16() / 8, torch.randn(64, 32, device="cuda").bfloat16()
    y = torch.randn(M, 64, device="cuda").bfloat16()
    out, t = hip_ops().lora_apply(y, x, A, B, 0.5)
    rows = torch.tensor([0, 1, M // 2, M - 65, M - 33, M - 1], device="cuda")
    ref = 0.5 * (t[rows].double() @ B.double().t()) + y[rows].double()
    assert (out[rows].double() - ref).norm() <= 2.0 ** -9 * 1.05 * ref.norm()


@pytest.mark.parametrize("M,H,O,R", [(1, 64, 64, 32), (8, 8192, 64, 64), (63, 192, 320, 32), (64, 256, 576, 64),
                                     (1000, 512, 4096, 32), (2113, 4096, 192, 64), (8192, 64, 12288, 32),
                                     (65, 320, 192, 8), (2000, 4096, 576, 16), (300, 64, 4096, 40)])
def test_adapter_grads(M, H, O, R):
    """Strips partly empty, parts of the rows and their ends, both ranks."""
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    x = torch.randn(M, H, device="cuda").bfloat16()
    A = (torch.randn(R, H, device="cuda") / H ** 0.5).bfloat16()
    B = (torch.randn(O, R, device="cuda") / R ** 0.5).bfloat16()
    y, g = (torch.randn(M, O, device="cuda").bfloat16() for _ in range(2))
    out, tt = hip_ops().lora_forward(y, x, A, B, 0.5)
    full = 32 if R <= 32 else 64
    A0, B0 = torch.zeros(full, H, device="cuda").bfloat16(), torch.zeros(O, full, device="cuda").bfloat16()
    A0[:R], B0[:, :R] = A, B                    # what is filled up with zeros
    out2, t = hip_ops().lora_apply(y, x, A0, B0, 0.5)
    assert torch.equal(out, out2) and torch.equal(tt[:, :M], t.t()) and not tt[:, M:].any()
    assert all(torch.equal(a, b) for a, b in zip(hip_ops().lora_apply(y, x, A, B, 0.5), (out, t)))
    da, db, dt, a_t = hip_ops().lora_grads(g, x, A, B, tt, 0.5)
    assert torch.equal(a_t, A0.t()) and not dt[:, R:].any()
    t, dt = t[:, :R], dt[:, :R]
    dtd = 0.5 * (g.double() @ B.double())
    for got, ref in ((dt, dtd), (da, dt.double().t() @ x.double()), (db, 0.5 * (g.double().t() @ t.double()))):
        # each value is rounded to bf16 once
        assert (got.double() - ref).norm() <= 2.0 ** -9 * 1.05 * ref.norm()


@pytest.mark.parametrize("T,N,K,R", [(200, 64, 64, 32), (300, 128, 320, 64), (1000, 192, 520, 32), (513, 1024, 256, 96),
                                     (1001, 6144, 1536, 32), (256, 8192, 264, 64), (4100, 256, 2048, 32)])
def test_input_grad_with_an_extra_product(T, N, K, R):
    """Tiles of every height, partly empty, and sums in parts: the extra product is in one of them."""
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    g, t = torch.randn(T, N, device="cuda").bfloat16(), torch.randn(T, R, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") / N ** 0.5).bfloat16()
    A = (torch.randn(R, K, device="cuda") / R ** 0.5).bfloat16()
    dx = hip_ops().linear_dx_extra(g, w, t, A.t().contiguous())
    ref = g.double() @ w.double() + t.double() @ A.double()
    assert (dx.double() - ref).norm() <= 2.0 ** -9 * 1.05 * ref.norm()


@pytest.mark.parametrize("rank", [8, 32, 48])
@pytest.mark.parametrize("T,K,N,need_x", [(2048, 2048, 2560, True), (2048, 2048, 2560, False), (64, 128, 192, True),
                                          (8, 64, 64, True), (0, 128, 192, True)])
def test_adapted_layer(T, K, N, need_x, rank):
    from automodel_amd.peft.lora import LinearLoRA

    torch.manual_seed(0)
    lin = LinearLoRA(torch.nn.Linear(K, N, bias=False), rank, 2.0 * rank).to("cuda", torch.bfloat16)
    torch.nn.init.normal_(lin.lora_B.weight, std=0.1)
    x = torch.randn(2, T // 2, K, device="cuda").bfloat16().requires_grad_(need_x)
    g = torch.randn(2, T // 2, N, device="cuda").bfloat16()
    wrt = [lin.lora_A.weight, lin.lora_B.weight, *([x] if need_x else [])]
    got = torch.autograd.grad(lin(x), wrt, g)
    again = torch.autograd.grad(lin(x), wrt, g, create_graph=True)        # torch's products
    w, a, b, xd, gd = (v.detach().double() for v in (lin.base.weight, lin.lora_A.weight, lin.lora_B.weight, x, g))
    xd, gd = xd.view(T, K), gd.view(T, N)
    dt = 2.0 * gd @ b
    for grads in (got, again):
        for v, ref in zip(grads, (dt.t() @ xd, 2.0 * gd.t() @ (xd @ a.t()), gd @ w + dt @ a)):
            # t and dt are rounded to bf16, some results a few times more
            assert (v.double().view(ref.shape) - ref).norm() <= 2.0 ** -8 * ref.norm()


@pytest.mark.parametrize("rank", [8, 32, 40])
def test_infinite_rows(rank):
    """They are infinite, and not NaN, where all signs agree, as the modules have them."""
    from automodel_amd.peft.lora import LinearLoRA

    torch.manual_seed(0)
    lin = LinearLoRA(torch.nn.Linear(128, 64, bias=False), rank, 2.0 * rank).to("cuda", torch.bfloat16)
    with torch.no_grad():
        for p in lin.parameters():
            p.copy_(torch.rand(p.shape) + 0.1)
    x, g = (torch.randn(16, n, device="cuda").bfloat16() for n in (128, 64))
    x[3, 70], x[5, 1], g[2, 7], g[9, 63] = float("inf"), -float("inf"), float("inf"), -float("inf")
    x.requires_grad_()
    y = lin(x)
    dx, = torch.autograd.grad(y, x, g)
    for got, rows in ((y, (3, 5)), (dx, (2, 9))):
        assert (got[rows[0]] == float("inf")).all() and (got[rows[1]] == -float("inf")).all()
        assert got.isfinite().all(1).sum() == 14
