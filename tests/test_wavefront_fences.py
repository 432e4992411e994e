"""Lanes of one wavefront that hand numbers to each other through LDS: the barrier of a wavefront orders instructions, not memory, so
a release stands before it and, where a lane then reads what another wrote, an acquire behind it (CPU)."""

import re

from shrike_amd.csrc.build import CSRC

RELEASE, BARRIER, ACQUIRE = ('__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");', "__builtin_amdgcn_wave_barrier();",
                             '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");')


def test_no_wavefront_barrier_without_its_fences():
    users = {}
    for path in sorted([*CSRC.glob("*.hip"), *CSRC.glob("*.h")]):
        lines = [line.strip() for line in path.read_text().splitlines()]
        for i, line in enumerate(lines):
            if BARRIER not in line:
                continue
            assert lines[i - 1] == RELEASE, (path.name, i + 1)
            if lines[i + 1] != ACQUIRE:  # then what follows writes
                rest = "\n".join(lines[i + 1 : i + 8])
                assert re.search(r"\w+\[[^\]]*\] = ", rest), (path.name, i + 1)
            users[path.name] = users.get(path.name, 0) + 1
    assert {"attention_mfma.hip", "attention_diff_mfma.hip", "moe_few.hip"} <= set(users)


def test_the_list_of_an_expert_is_read_behind_its_writes():
    text = (CSRC / "moe_few.hip").read_text()
    write, read = text.index("place[__popcll("), text.index("mine = place[")
    between = text[write:read]
    assert between.index(RELEASE) < between.index(BARRIER) < between.index(ACQUIRE)
