"""Which steps' float32 attention takes two neighbouring tokens a workgroup (CPU)."""

import pytest

from shrike_amd.parts.attention import f32_pairs

FAR = 1 << 40


@pytest.mark.parametrize("decodes, portions, kv_heads, dim, expected", [
    (0, [(0, 509)], 2, 64, True),
    (256, [], 2, 64, False), (256, [], 4, 128, False), (0, [], 2, 64, False),  # nobody has a neighbour
    (0, [(0, 1)] * 300, 4, 64, False),
    (0, [(0, 200)], 2, 64, True), (0, [(0, 25)] * 8, 2, 64, False), (0, [(0, 25)] * 16, 2, 64, True),
    (0, [(0, 25)] * 16, 4, 128, False), (0, [(0, 200)] * 4, 4, 128, False), (0, [(0, 300)] * 4, 4, 128, True),
    (0, [(1000, 25)] * 16, 4, 128, True),  # few tokens behind many
    (40, [(0, 500)], 4, 128, True), (200, [(0, 500)], 4, 128, False), (200, [(0, 500)], 4, 64, True), (600, [(0, 500)], 4, 64, False),
])
def test_by_neighbours_and_keys(decodes, portions, kv_heads, dim, expected):
    q_lens, starts = [1] * decodes + [n for _, n in portions], [700] * decodes + [at for at, _ in portions]
    assert f32_pairs(decodes, q_lens, starts, kv_heads, dim, FAR) is expected


def test_a_window_bounds_the_keys():
    args = (0, [600], [4000], 4, 128)
    assert f32_pairs(*args, FAR) and not f32_pairs(*args, 64)


def test_pairs_are_of_even_and_odd_tokens_of_the_step():
    # portions of two tokens that begin at odd ones: no token's partner is of its own sequence
    assert not f32_pairs(1, [1] + [2] * 400, [700] * 401, 4, 64, FAR)
    assert f32_pairs(2, [1, 1] + [2] * 400, [700] * 402, 4, 64, FAR)
