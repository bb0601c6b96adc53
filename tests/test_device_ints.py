"""Host integers on the device without a copy that waits."""

import pytest
import torch

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a GPU")]


@pytest.mark.parametrize("n", [0, 1, 2, 255, 256, 257, 959, 960, 961, 2500])
def test_values(n):
    from automodel_amd.ops._backend import hip_ops

    values = [(-1) ** i * (i * 7919 % (1 << 31)) for i in range(n)]
    out = hip_ops().device_ints(values, torch.device("cuda"))
    assert out.dtype == torch.int32 and out.tolist() == values


def test_out_of_range():
    from automodel_amd.ops._backend import hip_ops

    assert hip_ops().device_ints([-2 ** 31, 2 ** 31 - 1], torch.device("cuda")).tolist() == [-2 ** 31, 2 ** 31 - 1]
    with pytest.raises(RuntimeError):
        hip_ops().device_ints([2 ** 31], torch.device("cuda"))
