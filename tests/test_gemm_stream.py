"""Linear layers of 3 to 16 rows as streams of weights: edges of the row blocks, of the parts
of K and of the rows of x, and what stays with the general kernel."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(b, k, sizes, seed=0):
    g = torch.Generator("cuda").manual_seed(seed)
    x = torch.randn(b, k, generator=g, device="cuda").bfloat16()
    return x, [torch.randn(n, k, generator=g, device="cuda").bfloat16() for n in sizes]


def _close(y, want, x, w, out_eps=2.0**-8):
    # a float32 sum of K products, each below 2^-24 of the absolute sum off, then rounded once
    absolute = x.double().abs() @ w.double().abs().t()
    bound = out_eps * want.abs() + x.shape[1] * 2.0**-24 * absolute
    assert ((y.double() - want).abs() <= bound).all()


def _close_gated(y, x, ws, gate):
    u, k = x.double() @ ws[1].double().t(), x.shape[1]
    want = torch.nn.functional.silu(gate) * u
    # |d silu| <= 1.1, and the errors of both factors meet the other factor; __expf: 4 ulp
    err, err_u = (k * 2.0**-24 * (x.double().abs() @ w.double().abs().t()) for w in ws)
    bound = (2.0**-8 + 2.0**-18) * want.abs() + 1.1 * err * u.abs() + err_u * gate.abs()
    assert ((y.double() - want).abs() <= bound + 1e-30).all()


# one row, one less and one more than a block; K of 1 tile (fewer than
# waves), of tiles that the waves share unevenly, and of a multiple of 8192
@pytest.mark.parametrize("n,k", [(1, 128), (7, 384), (9, 1152), (2049, 1152), (5121, 1152), (6144, 128),
                                 (7169, 1408), (10239, 1152), (10241, 2176), (12287, 1152),
                                 (14335, 2176), (16385, 1152), (8191, 8192), (40, 14336)])
@pytest.mark.parametrize("b", [3, 8, 9, 16])
def test_rows(n, k, b):
    from automodel_amd.ops._backend import hip_ops

    x, (w,) = _operands(b, k, [n])
    want = x.double() @ w.double().t()
    _close(hip_ops().gemm_skinny_bf16(x, w, False, True, 0), want, x, w, 2.0**-24)
    _close(hip_ops().gemm_skinny_bf16(x, w, False, False, 0), want, x, w)


# every kernel that the rule has: rows of W a workgroup, slots of a ring, waves, at rows of W that
# are no multiple of them; gate and up share a workgroup's rows, so that from 24 on either's are no
# multiple of 16
@pytest.mark.parametrize("shape,n,k,bs", [
    ((8, 3, 8), 17, 640, (3, 8, 9, 16)), ((16, 1, 4), 18541, 128, (8,)), ((16, 2, 4), 17, 128, (3, 16)),
    ((16, 2, 8), 2083, 3200, (8, 16)), ((24, 1, 4), 8209, 128, (8, 16)), ((24, 2, 4), 4113, 128, (8, 16)),
    ((32, 1, 4), 12377, 128, (8, 9)), ((32, 2, 4), 6179, 128, (8, 16)), ((40, 1, 4), 18159, 2176, (8,)),
    ((40, 1, 4), 16547, 2176, (16,)), ((40, 2, 4), 8217, 2176, (8, 16)), ((48, 1, 4), 10301, 2176, (5, 16)),
    ((56, 1, 4), 12335, 2176, (8, 16)), ((64, 1, 4), 14579, 2176, (8, 16)),
])
@pytest.mark.parametrize("glu", [False, True])
def test_every_kernel(shape, n, k, bs, glu):
    from automodel_amd.ops._backend import hip_ops

    ops = hip_ops()
    n = n // 2 if glu and n > 17 else n            # so many of gate and of up
    for b in bs:
        assert ops.decode_rows_shape([n], k, b, glu) == shape
        x, ws = _operands(b, k, [n] * (2 if glu else 1))
        (y,) = ops.decode_rows(x, ws, glu, False, None)
        gate = x.double() @ ws[0].double().t()
        if glu:
            _close_gated(y, x, ws, gate)
        else:
            _close(y, gate, x, ws[0])


# several weights in one launch, with uneven ends
@pytest.mark.parametrize("sizes,k,shape", [((4099, 1027, 1029), 4096, (32, 2, 4)), ((6000, 1503, 1505), 4096, (40, 2, 4)),
                                           ((6000, 1503, 1505), 1152, (24, 1, 4)), ((8200, 2053, 2055), 4096, (56, 1, 4))])
@pytest.mark.parametrize("b", [8, 16])
def test_several_weights(sizes, k, shape, b):
    from automodel_amd.ops._backend import hip_ops

    assert hip_ops().decode_rows_shape(sizes, k, b) == shape
    x, ws = _operands(b, k, sizes)
    for y, w in zip(hip_ops().decode_rows(x, ws, False, False, None), ws):
        _close(y, x.double() @ w.double().t(), x, w)


@pytest.mark.parametrize("sizes,k", [((4096, 1024, 1024), 512), ((33, 1, 15), 1152)])
@pytest.mark.parametrize("b", [4, 13])
def test_segments_residual_and_gate(sizes, k, b):
    from automodel_amd.ops._backend import hip_ops

    x, ws = _operands(b, k, sizes)
    for y, w in zip(hip_ops().decode_rows(x, ws, False, False, None), ws):
        _close(y, x.double() @ w.double().t(), x, w)
    res = torch.randn(b, sizes[0], device="cuda").bfloat16()
    (y,) = hip_ops().decode_rows(x, ws[:1], False, False, res)
    want = x.double() @ ws[0].double().t() + res.double()
    _close(y, want, x, ws[0])
    up = ws[0].flip(0).contiguous()
    (y,) = hip_ops().decode_rows(x, [ws[0], up], True, False, None)
    _close_gated(y, x, [ws[0], up], x.double() @ ws[0].double().t())


@pytest.mark.parametrize("group,last", [(16, 16), (48, 16), (2048, 2048), (6144, 6144)])
def test_groups(group, last):
    from automodel_amd.ops._backend import hip_ops

    xs = torch.randn(2, 5, 256, device="cuda").bfloat16()
    w = torch.randn(group + last, 256, device="cuda").bfloat16()
    y = hip_ops().gemm_skinny_bf16(xs.view(10, 256), w, False, False, group)
    _close(y[:, :group], xs[0].double() @ w[:group].double().t(), xs[0], w[:group])
    _close(y[:, group:], xs[1].double() @ w[group:].double().t(), xs[1], w[group:])


def test_other_forms_keep_the_general_kernel():
    from automodel_amd.ops._backend import hip_ops

    for k, skip in ((136, 0), (256, 4)):           # K % 128; a weight that is not on 16 bytes
        x, (w,) = _operands(5, k, [70])
        flat = torch.empty(w.numel() + skip, device="cuda", dtype=w.dtype)
        moved = flat[skip:].view_as(w).copy_(w)
        y = hip_ops().gemm_skinny_bf16(x, moved, False, False, 0)
        _close(y, x.double() @ w.double().t(), x, w)
    # what lies beyond a weight's rows and x's rows does not reach the output
    x, (w,) = _operands(8, 256, [24])
    w[16:] = float("nan")
    x[5:] = float("inf")
    y = hip_ops().gemm_skinny_bf16(x[:5], w[:16], False, False, 0)
    _close(y, x[:5].double() @ w[:16].double().t(), x[:5], w[:16])
