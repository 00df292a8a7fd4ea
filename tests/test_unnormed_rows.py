"""Which 32-bit rows a product norms itself: only those whose norm has one aligned 32-bit weight a column (checked without a GPU)."""
import pytest
import torch

from xyntetik_runner_amd.csrc.ops import Ops, UnnormedRows


def aligned(n, dtype=torch.float32, by=0):
    room = torch.ones(n + 16, dtype=dtype)
    at = (-room.data_ptr() % 16) // room.element_size() + by
    return room[at:at + n]


@pytest.mark.parametrize("weight,taken", [(aligned(64), True), (aligned(60), False), (aligned(128), False), (aligned(64, torch.bfloat16), False),
                                          (aligned(64, by=1), False), (aligned(128)[::2], False), (None, False)])
def test_weight_of_the_norm(weight, taken):
    ops = Ops.__new__(Ops)
    ops.fold_norms, ops.EXTRA_ROWS = True, 4
    a, w = aligned(128).view(2, 64), aligned(96 * 64).view(96, 64)
    assert ops._extra_ok(a, w, None)
    assert ops._extra_ok(UnnormedRows(a, weight, 1e-5), w, None) == taken
