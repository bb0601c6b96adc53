"""The attention forward of long walks: ends of rows and keys, rows that see keys from the middle on,
sinks, negative scales, and scores that leave what the first keys' maximum allows."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _check(q, k, v, scale, causal, q_start=0, sink=None, ordered=None):
    """``ordered``: sixteens of rows a wave of the ordered kernel that the call has to come to."""
    from automodel_amd.ops._backend import hip_ops

    if ordered is not None:
        assert _ordered(q, k, causal, q_start) == ordered
    out, lse = hip_ops().flash_attn_fwd(q, k, v, scale, causal, q_start, None, sink)
    B, S, H, _ = q.shape
    n, rep = k.shape[1], H // k.shape[2]
    g = torch.Generator().manual_seed(1)
    some = torch.randint(S, (96,), generator=g).tolist()
    rows = torch.tensor(sorted({0, 1, S // 2, S - 2, S - 1, *some})).cuda().clamp(0, S - 1)
    for b, h in {(0, 0), (B - 1, H - 1), (0, H // 2)}:
        x, y = k[b, :, h // rep].double(), v[b, :, h // rep].double()
        s = q[b, rows, h].double() @ x.t() * scale
        if causal:
            s = s.masked_fill(torch.arange(n, device="cuda") > (rows + q_start)[:, None], float("-inf"))
        most = s.amax(-1, keepdim=True)
        p = (s - most).exp()
        total = p.sum(-1, keepdim=True)
        if sink is not None:
            total = total + (sink[h].double() - most).exp()
        p = p / total
        # the weights rounded once to bf16 and the output too: half a step of 8 significant bits,
        # up to 2^-8 of the value, each. A float32 score is 2^-24 a
        # product off its absolute sum, scale * log2(e) and the difference to the maximum once each
        # of the score itself; so much relative to a weight is the error of all of them
        of_score = (2.0**-24 * abs(scale) * (q.shape[-1] * (q[b, rows, h].double().abs() @ x.abs().t()))
                    ).amax(-1, keepdim=True) + 2.0**-22 * s.masked_fill(p == 0, 0).abs().amax(-1, keepdim=True)
        want, absolute = p @ y, p @ y.abs()
        bound = (2.0**-8 + 2 * of_score + 2.0**-16) * absolute * 1.02 + 2.0**-8 * want.abs() + 1e-30
        err = (out[b, rows, h].double() - want).abs()
        assert (err <= bound).all(), (err / bound).max()
        ref = (most + total.log()).squeeze(-1)
        assert ((lse[b, h, rows].double() - ref).abs() <= 2 * of_score.squeeze(-1) + 2.0**-16
                + 2.0**-22 * ref.abs()).all()


def _ordered(q, k, causal, q_start=0):
    from automodel_amd.ops._backend import hip_ops

    return hip_ops().flash_attn_fwd_ordered(*q.shape[:2], k.shape[1], q.shape[2], k.shape[2], q.shape[3], 128,
                                            causal, q_start)


def _inputs(B, S, n, H, K, D, seed=0):
    g = torch.Generator("cuda").manual_seed(seed)
    return tuple(torch.randn(B, m, h, d, generator=g, device="cuda").bfloat16()
                 for m, h, d in ((S, H, D), (n, K, D), (n, K, 128)))


# (ordered 0: not for these)
@pytest.mark.parametrize("B,S,n,H,K,D,causal,start,ordered", [
    (2, 1024, 1024, 32, 8, 128, False, 0, 4),
    (2, 997, 1500, 32, 8, 128, False, 0, 0),
    (1, 1024, 1501, 64, 8, 128, False, 0, 4),     # a short last tile of keys
    (1, 1793, 1793, 32, 8, 128, False, 0, 4),     # one row in the last workgroups
    (64, 1025, 1025, 4, 2, 128, False, 0, 0),     # and where that leaves a round too empty
    (1, 8000, 8000, 16, 4, 128, True, 0, 4),
    (1, 8001, 8003, 16, 4, 128, True, 2, 4),
    (1, 512, 512, 8, 8, 192, True, 0, 3),
    (2, 577, 577, 8, 8, 192, True, 0, 3),
    (1, 193, 1300, 8, 8, 192, True, 700, 3),
    (1, 191, 1300, 8, 8, 192, True, 700, 0),
    (1, 600, 777, 16, 16, 192, False, 0, 3),
    (2, 3001, 3001, 16, 16, 192, True, 0, 3),
    (1, 8192, 8192, 16, 16, 192, True, 0, 4),
    (2, 2047, 2050, 16, 16, 192, False, 0, 4),
])
def test_long_walks(B, S, n, H, K, D, causal, start, ordered):
    q, k, v = _inputs(B, S, n, H, K, D)
    _check(q, k, v, D**-0.5, causal, start, ordered=ordered)


@pytest.mark.parametrize("D,n,H", [(192, 700, 8), (128, 1100, 64)])
def test_sink_and_negative_scale(D, n, H):
    q, k, v = _inputs(1, n, n, H, H, D, 2)
    _check(q, k, v, -0.3, False, sink=torch.randn(H, device="cuda").bfloat16() * 4)
    _check(q, k, v, -0.3, D == 192, sink=torch.randn(H, device="cuda").bfloat16() * 4)


@pytest.mark.parametrize("D,H", [(192, 8), (128, 64)])
@pytest.mark.parametrize("kind", ["ramp", "late", "early", "first"])
def test_scores_far_above_the_first_ones(D, H, kind):
    n = 1024
    q, k, v = _inputs(1, n, n, H, H, D, 3)
    at = torch.arange(n, device="cuda")[:, None, None]
    factor = {"ramp": at / 16.0, "late": torch.where(at == 1000, 200.0, 1.0),
              "early": torch.where(at == 40, 200.0, 1.0), "first": torch.where(at == 3, 200.0, 1.0)}[kind]
    k = (k.float() * factor).bfloat16()
    _check(q, k, v, D**-0.5, False)
    if D == 192:
        _check(q, k, v, D**-0.5, True)


# (128, 128) has the ordered kernel for full rounds of workgroups without a mask, and for 8000 keys with one
@pytest.mark.parametrize("D,n,H,causal,ordered", [(128, 1024, 64, False, 4), (128, 8001, 16, True, 4), (192, 700, 8, True, 3),
                                                  (192, 700, 8, False, 3), (192, 2047, 32, False, 4)])
class TestOrdered:
    def test_sink_and_negative_scale(self, D, n, H, causal, ordered):
        q, k, v = _inputs(1, n, n, H, H, D, 4)
        _check(q, k, v, -0.3, causal, sink=torch.randn(H, device="cuda").bfloat16() * 4, ordered=ordered)

    def test_scale_of_zero(self, D, n, H, causal, ordered):
        q, k, v = _inputs(1, n, n, H, H, D, 5)
        _check(q, k, v, 0.0, causal, ordered=ordered)

    @pytest.mark.parametrize("kind", ["ramp", "late", "last"])
    def test_scores_far_above_the_first_ones(self, D, n, H, causal, ordered, kind):
        q, k, v = _inputs(1, n, n, H, H, D, 6)
        at = torch.arange(n, device="cuda")[:, None, None]
        factor = {"ramp": at * 64.0 / n, "late": torch.where(at == n - 100, 200.0, 1.0),
                  "last": torch.where(at == n - 1, 200.0, 1.0)}[kind]
        k = (k.float() * factor).bfloat16()
        _check(q, k, v, D**-0.5, causal, ordered=ordered)

    def test_nan_stays_in_its_rows(self, D, n, H, causal, ordered):
        from automodel_amd.ops._backend import hip_ops

        run = lambda q, k: hip_ops().flash_attn_fwd(q, k, v, D**-0.5, causal, 0, None, None)[0]
        q, k, v = _inputs(1, n, n, H, H, D, 7)
        assert _ordered(q, k, causal) == ordered
        clean = run(q, k)
        x = q.clone()
        x[0, 5, 0, 3] = float("nan")
        got = run(x, k)
        assert got[0, 5, 0].isnan().all()
        got[0, 5, 0] = clean[0, 5, 0]
        assert torch.equal(got, clean)
        for at in (3, n - 200):                     # among the first keys, and late
            x = k.clone()
            x[0, at, 1, 7] = float("nan")
            got, first = run(q, x), at if causal else 0       # the first row that sees it
            assert got[0, first:, 1].isnan().all() and torch.equal(got[0, :first], clean[0, :first])
            assert torch.equal(got[0, :, 2:], clean[0, :, 2:]) and torch.equal(got[0, :, 0], clean[0, :, 0])

    @pytest.mark.parametrize("hidden", [(40,), tuple(range(64)), tuple(range(1, 300))])
    def test_infinite_scores(self, D, n, H, causal, ordered, hidden):
        from automodel_amd.ops._backend import hip_ops

        q, k, v = _inputs(1, n, n, H, H, D, 8)
        assert _ordered(q, k, causal) == ordered
        q[..., 0] = 1.0
        k[:, list(hidden), :, 0] = float("-inf")     # keys that get no weight
        k[:, n - 150, 1, 0] = float("inf")           # and one in head 1 that leaves no number
        out = hip_ops().flash_attn_fwd(q, k, v, D**-0.5, causal, 0, None, None)[0]
        rows = torch.tensor(sorted({300, 301, n // 2, n - 151, n - 2, n - 1})).cuda()
        for h in (0, 1, H - 1):
            s = q[0, rows, h].double() @ k[0, :, h].double().t() * D**-0.5
            if causal:
                s = s.masked_fill(torch.arange(n, device="cuda") > rows[:, None], float("-inf"))
            p = s.softmax(-1)
            want, absolute = p @ v[0, :, h].double(), p @ v[0, :, h].double().abs()
            # weights and output rounded to bf16 once; float32 scores of some 10 are off by less than 2^-12
            bound = (2.0**-8 + 2.0**-12) * 1.02 * absolute + 2.0**-8 * want.abs()
            none = s.isposinf().any(-1)
            assert none.any() == (h == 1) and out[0, rows[none], h].isnan().all()
            assert ((out[0, rows, h].double() - want).abs() <= bound)[~none].all()
