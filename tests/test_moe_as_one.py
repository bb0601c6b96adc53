"""The expert layer as one function of autograd against one function for each of its parts."""

import pytest
import torch

from automodel_amd.moe.experts import GroupedExperts, fused_dispatch_combine

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


# hidden and inner widths on both sides of the rule, one expert, experts without tokens, one choice and nine, one token
@pytest.mark.parametrize("T,K,E,H,inter", [(1, 1, 1, 128, 128), (700, 2, 8, 512, 128), (333, 9, 40, 256, 128),
                                           (257, 3, 64, 256, 1408), (2000, 8, 16, 1024, 512)])
def test_gradients(T, K, E, H, inter):
    torch.manual_seed(T)
    experts = GroupedExperts(E, H, inter).to("cuda", torch.bfloat16)
    experts.init_weights(H ** -0.5)
    chosen = torch.rand(T, max(E - 2, 1), device="cuda").topk(K, -1)[1]        # the last two experts have no tokens
    probs = torch.rand(T, K, device="cuda").bfloat16().requires_grad_()
    x, d = (torch.randn(T, H, device="cuda").bfloat16() for _ in range(2))
    x.requires_grad_()
    inputs = [x, probs, *experts.parameters()]
    y = experts(x, probs, chosen)
    assert type(y.grad_fn).__name__ == "_ExpertsBackward"
    want = fused_dispatch_combine(x, probs, chosen, E, experts.forward_permuted)
    assert torch.equal(y, want)
    got = torch.autograd.grad(y, inputs, d, retain_graph=True)
    exact = [t.detach().double().requires_grad_() for t in inputs]
    out = torch.zeros(T, H, device="cuda", dtype=torch.float64)
    for e in range(E):
        rows, slot = (chosen == e).nonzero(as_tuple=True)
        h = torch.nn.functional.silu(exact[0][rows] @ exact[2][e].T) * (exact[0][rows] @ exact[3][e].T)
        out = out.index_add(0, rows, h @ exact[4][e].T * exact[1][rows, slot, None])
    exact = torch.autograd.grad(out, exact, d.double())
    for a, b, t in zip(got, torch.autograd.grad(want, inputs, d), exact):
        # up to eight roundings to 8 bits one after another (g, u, h, the weighted row, dh, dg or du, dx of the row and its
        # sum), each 2^-9 of the value at most; and no further from 64 bits than the parts, but for what chance does to
        # few values
        off = [float((v.double() - t).norm()) for v in (a, b)]
        assert a.dtype == b.dtype and off[0] <= 8 * 2.0 ** -9 * float(t.norm())
        assert off[0] <= off[1] * 1.05 + 2.0 ** -9 * float(t.norm()) * (t.numel() < 10000)
    for i in range(len(inputs)):            # one of them alone is the same
        (alone,) = torch.autograd.grad(y, [inputs[i]], d, retain_graph=True)
        assert torch.equal(alone, got[i])


def test_rows_of_the_activation():
    from automodel_amd.ops._backend import hip_ops

    for M, I in ((1, 8), (9, 264), (1000, 768)):
        torch.manual_seed(M)
        dh, g, u = (torch.randn(M, I, device="cuda").bfloat16() for _ in range(3))
        p, order = torch.rand(M, device="cuda"), torch.randperm(M, device="cuda").int()
        dg, du, ph, dp = hip_ops().swiglu_rows_bwd(dh, g, u, p, order)
        d, gd, ud = dh.double() * p.double()[:, None], g.double(), u.double()
        s = gd.sigmoid()
        for a, b in ((dg, d * ud * s * (1 + gd * (1 - s))), (du, d * gd * s), (ph, p.double()[:, None] * gd * s * ud)):
            # one rounding to 8 bits, and 32-bit arithmetic before it
            assert ((a.double() - b).abs() <= 2.0 ** -8 * b.abs() + 2.0 ** -20 * d.abs().max()).all()
        terms = dh.double() * gd * s * ud
        assert ((dp[order.long()].double() - terms.sum(1)).abs() <= 2.0 ** -20 * terms.abs().sum(1)).all()
    for bad in (lambda: hip_ops().swiglu_rows_bwd(dh, g, u[:, :-8], p, order), lambda: hip_ops().swiglu_rows_bwd(dh, g, u, p[:-1], order),
                lambda: hip_ops().swiglu_rows_bwd(dh.float(), g, u, p, order), lambda: hip_ops().swiglu_rows_bwd(dh, g, u, p, order.long())):
        with pytest.raises(RuntimeError):
            bad()


def test_what_stays_in_parts():
    def name(experts, T=8):
        x = torch.randn(T, experts.hidden_size, device="cuda").bfloat16().requires_grad_()
        probs, chosen = torch.rand(T, 2, device="cuda"), torch.zeros(T, 2, dtype=torch.long, device="cuda")
        return type(experts(x, probs, chosen).grad_fn).__name__

    def make(cls=GroupedExperts, H=256, inter=128):
        experts = cls(4, H, inter).to("cuda", torch.bfloat16)
        experts.init_weights()
        return experts

    class Other(GroupedExperts):
        def forward_permuted(self, x_perm, counts):
            return super().forward_permuted(x_perm, counts) * 2

    assert name(make()) == "_ExpertsBackward"
    own = make()
    own.forward_permuted = lambda x, counts: x
    eight = make()
    eight.fp8 = True
    for experts in (make(Other), own, eight, make(inter=72), make(H=264)):
        assert name(experts) == "_CombineWithProbsBackward"
