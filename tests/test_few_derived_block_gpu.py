"""A block derived from the pre-norm one that adds to the stream behind its parts: what it adds reaches the next block, in steps of few tokens as
in others."""

from dataclasses import dataclass, replace
from typing import ClassVar

import pytest
import torch

from .test_parts_gpu import cpu_weights, make_runner, small_spec, step_whole

pytestmark = pytest.mark.gpu


def derived_spec():
    from shrike_amd.config import BlockSpec
    from shrike_amd.kernels import ops
    from shrike_amd.parts.base import register_block
    from shrike_amd.parts.block import PreNormResidualBlock

    @dataclass(frozen=True)
    class ShiftedBlockSpec(BlockSpec):
        kind: ClassVar[str] = "toy_shifted"

    class ShiftedBlock(PreNormResidualBlock):
        def forward(self, ctx, hidden, cache):
            super().forward(ctx, hidden, cache)
            hidden.settle(ctx)
            ops.add_rows(hidden.resid, None, self.shift)

        def load(self, tensors, runtime):
            super().load(tensors, runtime)
            self.shift = 2.0 * torch.cos(torch.arange(self.width, device=runtime.device, dtype=torch.float32))

    register_block(ShiftedBlockSpec.kind, ShiftedBlock)
    spec = small_spec()
    first, second = spec.blocks
    return replace(spec, blocks=(ShiftedBlockSpec(first.name, first.mixer, first.ffn, first.mixer_norm, first.ffn_norm), second))


@pytest.mark.parametrize("n", [5, 16])
def test_what_a_derived_block_adds_is_not_lost(n, monkeypatch):
    from shrike_amd.kernels import ops

    spec = derived_spec()
    weights, ids = cpu_weights(spec), [(7 * i + 3) % 97 for i in range(n)]
    runner, _, cache = make_runner(spec, weights, torch.bfloat16)
    got = step_whole(runner, cache, ids)
    monkeypatch.setattr(ops, "few_stream_sums", lambda *sizes: 0)  # (the products and norms of other steps)
    runner, _, cache = make_runner(spec, weights, torch.bfloat16)
    want = step_whole(runner, cache, ids)
    assert float((got - want).norm() / want.norm()) < 0.02  # (two layers of bfloat16)
