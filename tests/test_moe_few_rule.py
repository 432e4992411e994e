"""Which layers' experts run in the kernels for up to 16 tokens: those whose empty workgroups cost less than the launches they spare (CPU)."""

import pytest

from shrike_amd.kernels import ops


@pytest.mark.parametrize("width, ff, shared, experts, top, identity, few", [
    (3584, 4736, 9472, 8, 2, 2, True), (896, 1216, 2432, 8, 2, 2, True), (896, 1216, 2432, 16, 2, 0, True), (3584, 4736, 9472, 16, 8, 0, True),
    (64, 64, 0, 8, 2, 0, True), (64, 64, 64, 64, 2, 0, True), (512, 512, 512, 16, 2, 0, True), (4096, 4096, 0, 8, 2, 0, True),
    (896, 1216, 2432, 64, 2, 0, False), (2048, 768, 0, 128, 8, 0, False), (2048, 768, 0, 512, 8, 0, False), (7168, 2048, 2048, 256, 8, 0, False),
    (512, 512, 0, 16, 2, 0, False), (2048, 512, 512, 64, 8, 0, False), (64, 64, 0, 512, 1, 0, False), (4096, 256, 256, 32, 8, 0, False),
    (64, 64, 0, 8, 9, 8, False), (64, 64, 0, 4, 5, 0, False)])
def test_by_sizes(width, ff, shared, experts, top, identity, few):
    assert ops.moe_few_faster(width, ff, experts, top, shared, identity) is few
