"""Which kernel a call takes, by its sizes alone."""

import pytest

from automodel_amd.ops._backend import hip_ops, ops_available

pytestmark = pytest.mark.skipif(not ops_available(), reason="the library is not built")


@pytest.mark.parametrize("b", [3, 8, 9, 16])
def test_few_row_linears(b):
    def shape(n, k, glu=False):
        return hip_ops().decode_rows_shape([n], k, b, glu)

    # 8 rows of W in a ring that has the CU to itself: one workgroup a CU, a tile of K for each wave
    assert shape(2048, 4096)[0] == shape(1024, 4096, True)[0] == 8
    for n, k in ((4224, 768), (2049, 1024), (1232, 512), (17, 128)):
        assert shape(n, k)[0] > 8 and shape(n // 2 + 1, k, True)[0] > 8
    # several workgroups a CU share it: one slot where two leave no room, or where rows are short
    assert shape(28864, 3072)[:2] in ((40, 1), (48, 1), (56, 1), (64, 1))
    for n in (14400, 16384, 40960):
        for k in (512, 1024, 2048):
            assert shape(n, k)[1] == 1
    # rows of few columns leave no tiles for the waves of many rows of W
    assert shape(12032, 1280)[0] <= 32


@pytest.mark.parametrize("rows", [320, 384, 511])
def test_row_tiles_of_experts(rows):
    from automodel_amd.ops.grouped_gemm import tile_rows

    # the larger tile where it fills the chip with both products of a layer, else from 512 rows on
    for experts, inter, hidden, large in ((8, 2048, 4096, False), (4, 4096, 4096, rows == 511), (16, 768, 2048, False),
                                          (8, 14336, 4096, rows != 511), (64, 1408, 2048, rows > 330),
                                          (128, 768, 2048, rows > 330), (128, 2048, 2048, True)):
        assert tile_rows(rows * experts, experts, inter, hidden) == (256 if large else 128)
        assert tile_rows(319 * experts, experts, inter, hidden) == 128
        assert tile_rows(512 * experts, experts, inter, hidden) == 256


def test_attention_backward():
    def ordered(*sizes, causal=True, docs=0):
        return hip_ops().flash_attn_bwd_ordered(*sizes, causal, docs)

    for dims, tokens in (((128, 128), 256), ((192, 128), 192)):
        # short documents have the kernels before, for the heads of a group together; long ones, and
        # an unknown number of them, the ordered dK/dV; dQ of documents is never ordered
        for heads, group in ((32, 1), (8, 4)):
            most = 8192 * group // tokens
            assert ordered(1, 8192, 8192, 32, heads, *dims, docs=most) == (True, False)
            assert ordered(1, 8192, 8192, 32, heads, *dims, docs=most + 1) == (False, False)
        assert ordered(1, 8192, 8192, 32, 32, *dims, docs=-1) == (True, False)
        # few queries; long walks
        assert ordered(8, 64, 4096, 32, 32, *dims, causal=False) == (False, False)
        assert ordered(8, 4096, 4096, 32, 32, *dims) == (True, True)
    assert ordered(8, 4096, 4096, 32, 32, 64, 64) == ordered(8, 4096, 4096, 32, 32, 256, 256) == (False, False)


def test_attention_forward():
    def rows(S, heads, d, causal, B=1):
        return hip_ops().flash_attn_fwd_ordered(B, S, S, heads, heads, d, 128, causal)

    # without a mask full rounds of workgroups of 256 rows, counted in rows: 7 x 256 for 1672 are not
    assert rows(1024, 64, 128, False) == rows(7103, 8, 128, False) == 4
    assert rows(1672, 128, 128, False) == rows(1672, 32, 128, False, 4) == rows(5000, 32, 128, False) == 0
    # with one: the last of three rounds begins with its longest workgroup
    assert rows(3001, 32, 192, True) == 3 and rows(3465, 32, 192, True) == 4
    assert rows(2048, 32, 192, True) == 3 and rows(2048, 48, 192, True) == 0
    assert rows(8192, 16, 192, True) == 4 and rows(16384, 32, 128, True) == 4 and rows(6000, 32, 128, True) == 0
