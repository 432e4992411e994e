"""Experts' products whose tiles leave a die from none to a whole round of workgroups at the end: halves of tiles where they fill no more
than half of it, also halves that lie beyond the matrix, against float64."""

import pytest

from tests import test_moe_tiles_gpu as lists

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form, each", [("bounded", each) for each in (16, 17, 31, 32, 33, 48, 49)] + [("single", 31), ("single", 33)])
def test_tiles_beyond_the_last_whole_round(form, each):
    """`each` tiles a die of the first product: 192 features in two tiles of 128 (half of the second's are none), in one of 256 without a gate."""
    from shrike_amd.kernels import ops

    width, ff, single = 128, 192, form == "single"
    count = 8 * each * 128 // (1 if single else 2) - 70
    assert ops.moe_experts_tiles(count, width, ff, 1, 2, 1, single)[0] == (256, 128)
    lists.test_lists_of_every_length(width, ff, [count], form)
