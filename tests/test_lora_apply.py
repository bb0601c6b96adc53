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
