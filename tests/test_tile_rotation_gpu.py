"""Tiles that rotate what they write: cosines and sines in LDS for all rows, for 32 rows of each wave, or from memory; values whose
aligned groups of positions begin at any row."""
import pytest

from test_kernels_gpu import check_projection_with_rotation_and_cache_write, ops      # noqa: F401  (ops is the fixture)

pytestmark = pytest.mark.gpu


# 12, 14, 26: eight waves, four of them along rows (a table of 32 rows of each: up to 128 x 1 KB do not fit); 17, 27: four waves (all
# rows' table of 128 channels fits, of 256 a part); 29: one wave along rows.  Odd numbers of pairs, whose table is copied
# pair by pair, and heads that are rotated in part of 16 columns.
@pytest.mark.parametrize("variant", [12, 14, 17, 26, 27, 29])
@pytest.mark.parametrize("H,Hk,D,rot,inter,ps", [(3, 1, 128, 128, False, 16), (2, 1, 256, 256, False, 8), (1, 1, 256, 254, True, 16), (3, 2, 48, 18, True, 4),
                                                 (2, 1, 64, 6, True, 16), (2, 2, 96, 16, False, 32), (2, 1, 64, 0, False, 16)])
def test_tables_and_row_groups(ops, variant, H, Hk, D, rot, inter, ps):      # noqa: F811
    check_projection_with_rotation_and_cache_write(ops, "bfloat16", H, Hk, D, rot, inter, ps, [3, 0, 7], [257, 11, 250], D == 96, 256, variant=variant)
