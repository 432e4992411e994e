"""Which run's last product may add to the stream for the next run's norm: nothing may come between them (CPU)."""

from dataclasses import dataclass, replace
from typing import ClassVar

import pytest

from shrike_amd.config import BlockSpec, ScheduleEntry
from shrike_amd.config.specs import ParallelBlockSpec
from shrike_amd.models import DecoderModel
from shrike_amd.parts.base import register_block
from shrike_amd.parts.block import PreNormResidualBlock

from .test_parts_gpu import small_spec


@dataclass(frozen=True)
class DerivedBlockSpec(BlockSpec):
    kind: ClassVar[str] = "toy_derived"


class DerivedBlock(PreNormResidualBlock):
    def forward(self, ctx, hidden, cache):
        super().forward(ctx, hidden, cache)
        hidden.settle(ctx)


register_block(DerivedBlockSpec.kind, DerivedBlock)


def following(blocks=None, **changes):
    spec = small_spec(**changes)
    if blocks is not None:
        spec = replace(spec, blocks=blocks(spec.blocks))
    model = DecoderModel(spec)
    return [None if f is None else f == (model.blocks[e.block].mixer_norm, model.blocks[e.block].mixer)
            for f, e in zip(model._following, [*spec.schedule[1:], spec.schedule[0]])]


def derived(block):
    return DerivedBlockSpec(block.name, block.mixer, block.ffn, block.mixer_norm, block.ffn_norm)


def parallel(block):
    return ParallelBlockSpec(block.name, norm=block.mixer_norm, mixer=block.mixer, ffn=block.ffn)


@pytest.mark.parametrize("case, expected", [
    (dict(), [True, None]),
    (dict(schedule=(ScheduleEntry(0), ScheduleEntry(1), ScheduleEntry(0, cache_of=0))), [True, True, None]),
    (dict(schedule=(ScheduleEntry(0), ScheduleEntry(1, add_embedding=True))), [None, None]),
    (dict(schedule=(ScheduleEntry(0), ScheduleEntry(1, add_vector=("rows", 1))), stream_vectors=(("rows", 2),)), [None, None]),
    (dict(blocks=lambda b: (derived(b[0]), b[1])), [None, None]),  # the run itself
    (dict(blocks=lambda b: (b[0], derived(b[1]))), [None, None]),  # the next one
    (dict(blocks=lambda b: (b[0], parallel(b[1]))), [None, None]),
    (dict(blocks=lambda b: (parallel(b[0]), b[1])), [None, None])])
def test_nothing_may_come_between(case, expected):
    assert following(**case) == expected
