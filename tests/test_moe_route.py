"""Device-side routing plan, the combine's backward and the two-pair dx."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (3, 2, 5), (64, 4, 64), (257, 8, 128), (1000, 6, 300), (40, 2, 4096),
                                   (9000, 8, 128), (33, 3, 1025)])
def test_route_plan(T, K, E):
    from automodel_amd.ops._backend import hip_ops

    g = torch.Generator().manual_seed(T)
    idx = torch.rand(T, E, generator=g).topk(K, -1)[1].cuda()
    probs = torch.rand(T, K, generator=g).cuda()
    counts, order, src, pos, perm_probs = hip_ops().route_plan(idx, probs, E)
    flat = idx.reshape(-1)
    want = flat.argsort(stable=True)
    assert torch.equal(order.long(), want)
    assert torch.equal(counts.long(), torch.bincount(flat, minlength=E))
    assert torch.equal(src.long(), want // K)
    assert torch.equal(pos.reshape(-1).long()[want], torch.arange(T * K, device="cuda"))
    assert torch.equal(perm_probs, probs.reshape(-1)[want])


@pytest.mark.parametrize("T,K,H", [(1, 1, 8), (37, 3, 520), (100, 8, 2048)])
def test_combine_backward(T, K, H):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    idx = torch.rand(T, 16).topk(K, -1)[1].cuda()
    probs = torch.rand(T, K, device="cuda")
    _, order, src, _, p = hip_ops().route_plan(idx, probs, 16)
    g = torch.randn(T, H, device="cuda").bfloat16()
    y = torch.randn(T * K, H, device="cuda").bfloat16()
    dy, dp = hip_ops().combine_bwd(g, y, src, order, p)
    gp = g.float()[src.long()]
    assert torch.equal(dy, (gp * p[:, None]).bfloat16())
    want = torch.empty(T * K, device="cuda", dtype=torch.float64)
    want[order.long()] = (gp.double() * y.double()).sum(-1)
    # H products summed in f32
    assert (dp.double() - want).abs().max() <= 2.0 ** -23 * H ** 0.5 * 4 * (gp.abs() * y.float().abs()).sum(-1).max()


@pytest.mark.parametrize("counts,N,K", [([5, 0, 130, 300], 128, 256), ([600, 0, 520], 1408, 128)])
@pytest.mark.parametrize("bm", [128, 256])
def test_two_pairs(counts, N, K, bm):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    M, E = sum(counts), len(counts)
    g1, g2 = (torch.randn(M, N, device="cuda").bfloat16() for _ in range(2))
    w1, w2 = (torch.randn(E, N, K, device="cuda").bfloat16() for _ in range(2))
    plan = hip_ops().build_group_plan(torch.tensor(counts, dtype=torch.int32, device="cuda"), M, bm)
    dx = hip_ops().grouped_gemm_nn2(g1, w1, g2, w2, *plan, bm)
    at = torch.tensor([0, *counts]).cumsum(0).tolist()
    want = torch.cat([g1[s].double() @ w1[e].double() + g2[s].double() @ w2[e].double()
                      for e, s in enumerate(slice(a, b) for a, b in zip(at, at[1:]))])
    assert (dx.double() - want).norm() <= 2.0 ** -9 * 1.02 * want.norm()


@pytest.mark.parametrize("T,E,K", [(1, 1, 1), (3, 63, 2), (5, 64, 32), (130, 65, 6), (4, 128, 8), (7, 129, 5),
                                   (2, 257, 8), (6, 512, 32), (33, 512, 1), (9, 8, 8), (0, 16, 2),
                                   (5, 40, 33), (5, 513, 4)])       # the last two: torch's own
def test_route_choice(T, E, K):
    from automodel_amd.moe.layers import _expert_load, _largest

    g = torch.Generator().manual_seed(E)
    s = torch.rand(T, 2 * E, generator=g).cuda()[:, ::2] - 0.5      # no two equal, not contiguous
    idx = _largest(s, K)
    assert torch.equal(idx, s.topk(K, dim=-1)[1])
    assert torch.equal(_expert_load(idx, E), torch.bincount(idx.reshape(-1), minlength=E).float())


def test_route_choice_of_special_values():
    from automodel_amd.moe.layers import _expert_load, _largest

    inf, nan = float("inf"), float("nan")
    s = torch.tensor([[-inf, 1.0, -inf, inf, -0.5], [0.0, nan, 2.0, -inf, inf], [3.0, 3.0, 3.0, 4.0, 3.0],
                      [-inf] * 5, [torch.finfo(torch.float32).min, -inf, 1e-45, 0.0, -1e-45]]).cuda()
    want = [[3, 1, 4, 0], [1, 4, 2, 0], [3, 0, 1, 2], [0, 1, 2, 3], [2, 3, 4, 0]]    # equal: the lowest first
    assert _largest(s, 4).tolist() == want
    many = torch.randint(0, 4096, (4097, 3), device="cuda")
    assert torch.equal(_expert_load(many.T, 4096), torch.bincount(many.reshape(-1), minlength=4096).float())


@pytest.mark.parametrize("T,H,E", [(1, 128, 8), (17, 640, 24), (33, 256, 64), (129, 1024, 72), (8200, 128, 128),
                                   (2500, 256, 128), (4100, 128, 40), (1000, 384, 16)])
def test_router_linear(T, H, E):
    from automodel_amd.moe.layers import _router_scores

    torch.manual_seed(T)
    x = torch.randn(T, 2 * H, device="cuda").bfloat16()[:, :H].requires_grad_()        # rows apart
    w = torch.randn(E * H + 1, device="cuda").bfloat16()[1:].view(E, H).requires_grad_()    # off a boundary
    d = torch.randn(T, E, device="cuda") * torch.logspace(-9, 3, E, device="cuda")
    y = _router_scores(x, w)
    assert y.grad_fn.name() == "_RouterLinearBackward" and y.dtype == torch.float32
    dx, dw = torch.autograd.grad(y, (x, w), d)
    x64, w64, d64 = x.detach().double(), w.detach().double(), d.double()

    def near(got, a, b, n):      # n products summed in f32 in any order, then the output's rounding
        want, size = a @ b, a.abs() @ b.abs()
        ulp = 2.0 ** -8 if got.dtype == torch.bfloat16 else 2.0 ** -23
        assert ((got.double() - want).abs() <= ulp * want.abs() + n * 2.0 ** -24 * size).all()

    near(y, x64, w64.t(), H)
    near(dx, d64, w64, 3 * E)
    near(dw, d64.t(), x64, 3 * T)


def test_router_linear_gradients_of_gradients():
    from automodel_amd.moe.layers import _router_scores

    torch.manual_seed(0)
    x = torch.randn(5, 128, device="cuda").bfloat16().requires_grad_()
    w = torch.randn(8, 128, device="cuda").bfloat16().requires_grad_()

    def twice(f):
        (dx,) = torch.autograd.grad(f(x, w).square().sum(), x, create_graph=True)
        return torch.autograd.grad(dx.float().square().sum(), w)[0].double()

    got, want = twice(_router_scores), twice(lambda a, b: torch.nn.functional.linear(a.float(), b.float()))
    assert (got - want).norm() <= 2.0 ** -7 * want.norm()      # two roundings to bf16 on each side
    # each part only where it is wanted; not finite stays not finite
    y = _router_scores(x.detach(), w)
    assert torch.equal(torch.autograd.grad(y, w, torch.full_like(y, float("inf")))[0].isfinite().any(),
                       torch.tensor(False, device="cuda"))
    assert _router_scores(x.detach(), w.detach()).grad_fn is None


@pytest.mark.parametrize("bad", [-1, 8, 2 ** 40])
def test_experts_that_do_not_exist_are_refused(bad):
    from automodel_amd.moe.config import MoEConfig
    from automodel_amd.moe.experts import GroupedExperts
    from automodel_amd.moe.layers import MoE
    from automodel_amd.moe.router_replay import RouterReplay, router_replay_context

    torch.manual_seed(0)
    x = torch.randn(4, 128, device="cuda").bfloat16()
    idx = torch.arange(8, device="cuda").view(4, 2)
    probs = torch.rand(4, 2, device="cuda")
    experts = GroupedExperts(8, 128, 128).to("cuda", torch.bfloat16)
    experts.init_weights()
    good = experts(x, probs, idx)
    assert torch.equal(experts(x, probs, idx, checked=True), good)
    idx[3, 1] = bad
    with pytest.raises(RuntimeError):
        experts(x, probs, idx)
    moe = MoE(128, MoEConfig(n_routed_experts=8, n_activated_experts=2, moe_intermediate_size=128)) \
        .to("cuda", torch.bfloat16)
    rr = RouterReplay()
    rr.records = [idx]
    with router_replay_context(rr), pytest.raises(RuntimeError):
        rr.start_replay()
        moe(x.view(1, 4, 128))


def test_a_routers_own_choice_is_not_waited_for(monkeypatch):
    from automodel_amd.moe import experts, layers
    from automodel_amd.moe.config import MoEConfig

    def fail(*_):
        raise AssertionError("looked at")

    monkeypatch.setattr(experts, "check_experts", fail)
    monkeypatch.setattr(layers, "check_experts", fail)
    for balanced in (False, True):
        moe = layers.MoE(128, MoEConfig(n_routed_experts=8, n_activated_experts=2, moe_intermediate_size=128,
                                        fake_balanced_gate=balanced)).to("cuda", torch.bfloat16)
        moe.experts.init_weights()
        moe(torch.randn(1, 4, 128, device="cuda").bfloat16())


@pytest.mark.parametrize("T,K,E", [(1, 1, 1), (3, 2, 5), (1025, 6, 64), (64, 8, 128), (37, 32, 300), (130, 4, 512)])
@pytest.mark.parametrize("softmax", [True, False])
@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_route_weights(T, K, E, softmax, norm, dtype):
    from automodel_amd.moe.layers import _chosen_weights, _RouteWeights

    torch.manual_seed(0)
    logits = (torch.randn(T, E, device="cuda") * 3).requires_grad_()
    idx = logits.detach().topk(K, -1)[1]
    g = torch.randn(T, K, device="cuda").to(dtype)
    act = lambda t: t.softmax(-1) if softmax else t.sigmoid()
    probs = _RouteWeights.apply(logits, act(logits.detach()), idx, softmax, norm, 2.5, dtype)
    assert probs.dtype == dtype
    d, = torch.autograd.grad(probs, logits, g, retain_graph=True)
    with_graph, = torch.autograd.grad(probs, logits, g, create_graph=True)
    batched, = torch.autograd.grad(probs, logits, torch.stack([g, 2 * g]), is_grads_batched=True)
    ld = logits.detach().double().requires_grad_()
    want = _chosen_weights(act(ld), idx, norm, 2.5, torch.float64)
    wd, = torch.autograd.grad(want, ld, g.double(), create_graph=True)
    # float32 sums of up to 512 terms; weights are rounded to bf16 once
    near = 2.0 ** -20
    assert ((probs.double() - want).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else near) * want.abs() + 1e-30).all()
    room = near * (float(wd.detach().abs().max()) + float(g.abs().max()))
    for got in (d, with_graph, batched[0], batched[1] / 2):
        assert (got.double() - wd).abs().max() <= room
    if E > 1:                                   # twice
        v = torch.randn_like(logits)
        second, = torch.autograd.grad(with_graph, logits, v)
        wanted, = torch.autograd.grad(wd, ld, v.double())
        assert (second.double() - wanted).abs().max() <= 64 * near * (float(wanted.detach().abs().max()) + float(g.abs().max()))


@pytest.mark.parametrize("options", [dict(), dict(score_func="sigmoid", expert_bias=True, route_scale=2.5),
                                     dict(norm_topk_prob=False), dict(aux_loss_coeff=0.01),
                                     dict(n_expert_groups=4, n_limited_groups=2), dict(topk_then_softmax=True)])
def test_gate_of_both_kinds(options, monkeypatch):
    """The gate with its kernels and with torch's operations."""
    from automodel_amd.moe import layers
    from automodel_amd.moe.config import MoEConfig

    torch.manual_seed(0)
    cfg = MoEConfig(n_routed_experts=16, n_activated_experts=4, moe_intermediate_size=64, **options)
    gate = layers.Gate(256, cfg).cuda().bfloat16()
    torch.nn.init.normal_(gate.weight, std=0.1)
    x = torch.randn(300, 256, device="cuda").bfloat16().requires_grad_()
    g = torch.randn(300, 4, device="cuda").bfloat16()

    def run():
        probs, idx = gate(x)
        loss = (probs * g).float().sum() + (gate.last_aux_loss if options.get("aux_loss_coeff") else 0)
        return (probs, idx, *torch.autograd.grad(loss, (x, gate.weight)))

    got = run()
    monkeypatch.setattr(layers, "_weighs", lambda *a: False)
    want = run()
    assert torch.equal(got[1], want[1])
    for a, b in zip((got[0], *got[2:]), (want[0], *want[2:])):
        # sums in another order before one rounding to bf16
        assert (a.float() - b.float()).norm() <= 2.0 ** -8 * b.float().norm()


@pytest.mark.parametrize("T,K,H", [(1, 1, 8), (37, 3, 520), (100, 8, 2048), (65, 6, 264), (9, 2, 4096), (20, 4, 16),
                                   (33, 5, 264), (17, 7, 128), (12, 9, 64), (5, 16, 40)])
def test_copies_combine_and_sum(T, K, H):
    from automodel_amd.ops._backend import hip_ops

    torch.manual_seed(0)
    idx = torch.rand(T, 16).topk(K, -1)[1].cuda()
    probs = torch.rand(T, K, device="cuda")
    pos = hip_ops().route_plan(idx, probs, 16)[3]
    x = torch.randn(T, H, device="cuda").bfloat16()
    copies = hip_ops().permute_rows(x, pos)
    assert torch.equal(copies[pos.long()], x[:, None].expand(T, K, H))
    y = torch.randn(T * K, H, device="cuda").bfloat16()
    rows = y[pos.long()].double()
    for got, want in ((hip_ops().unpermute_combine(y, pos, probs), (rows * probs[..., None]).sum(1)),
                      (hip_ops().unpermute_sum(y, pos), rows.sum(1))):
        # sums of K products in f32, rounded to bf16 once
        assert ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -20 * rows.abs().sum(1)).all()
