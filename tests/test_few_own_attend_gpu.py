"""A mixer derived from paged attention whose attend() reads the step's own keys and values: they stand beside the queries, in steps of few
tokens as in others."""

from dataclasses import dataclass, replace
from typing import ClassVar

import pytest
import torch

from .test_parts_gpu import cpu_weights, make_runner, small_spec, step_whole

pytestmark = pytest.mark.gpu


def spec_with_own_attend(seen):
    from shrike_amd.config import AttentionSpec
    from shrike_amd.parts.attention import PagedAttention
    from shrike_amd.parts.base import register_mixer

    @dataclass(frozen=True)
    class SeeingSpec(AttentionSpec):
        kind: ClassVar[str] = "toy_seeing_attention"

    class Seeing(PagedAttention):
        def attend(self, ctx, qkv, out, tables, cache):
            seen.append(qkv[:, self.spec.num_heads * self.spec.head_dim :].clone())
            super().attend(ctx, qkv, out, tables, cache)

    register_mixer(SeeingSpec.kind, Seeing)
    spec = small_spec()
    m = spec.blocks[0].mixer
    mixer = SeeingSpec(num_heads=m.num_heads, num_kv_heads=m.num_kv_heads, head_dim=m.head_dim, qkv_bias=m.qkv_bias, out_bias=m.out_bias,
                       scale=m.scale, position=m.position)
    return replace(spec, blocks=tuple(replace(b, mixer=mixer) for b in spec.blocks))


@pytest.mark.parametrize("n", [1, 9, 16])
def test_the_steps_values_stand_beside_its_queries(n, monkeypatch):
    from shrike_amd.kernels import ops

    seen = []
    spec = spec_with_own_attend(seen)
    weights, ids = cpu_weights(spec), [(7 * i + 3) % 97 for i in range(n)]
    for few in (True, False):
        if not few:
            monkeypatch.setattr(ops, "few_heads_takes", lambda *sizes: False)
        runner, _, cache = make_runner(spec, weights, torch.bfloat16)
        runner.use_graphs = runner.use_call_lists = False
        step_whole(runner, cache, ids)
    half = len(seen) // 2
    assert half == 2
    for got, want in zip(seen[:half], seen[half:]):  # (values as they were projected; keys before or behind their rotation)
        assert torch.equal(got[:, 32:], want[:, 32:]) and got.shape == (n, 64)
