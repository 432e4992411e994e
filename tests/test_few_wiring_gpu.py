"""Who adds to the stream, who divides by the root mean square and who rotates what it forms, in whole steps of few tokens: the
launches of two layers that allow it and of those that do not, and their logits beside the same steps of products and norms in kernels
of their own."""

from dataclasses import replace

import pytest
import torch

from .test_parts_gpu import cpu_weights, make_runner, small_spec, step_whole

pytestmark = pytest.mark.gpu

NAMES = ("few_stream", "few_gated", "few_heads")


def changed(spec, index, **changes):
    blocks = list(spec.blocks)
    blocks[index] = replace(blocks[index], **changes)
    return replace(spec, blocks=tuple(blocks))


def case(name):
    from shrike_amd.config.specs import LayerNormSpec, MoESpec, ParallelBlockSpec, RotarySpec, ScheduleEntry, SwiGLUSpec

    spec = small_spec()
    first, second = spec.blocks
    layernorm = LayerNormSpec(eps=1e-5)
    if name == "scaled residual":
        return changed(changed(spec, 0, residual_scale=0.5), 1, residual_scale=0.5)
    if name == "embedding again":
        return replace(spec, schedule=(ScheduleEntry(0), ScheduleEntry(1, add_embedding=True)))
    if name == "vector":
        return replace(spec, schedule=(ScheduleEntry(0), ScheduleEntry(1, add_vector=("rows", 1))), stream_vectors=(("rows", 2),))
    if name == "average":
        return replace(spec, schedule=(ScheduleEntry(0, depth_average="a0"), ScheduleEntry(1, depth_average="a1")))
    if name == "parallel block":
        return replace(spec, blocks=(first, ParallelBlockSpec(second.name, norm=second.mixer_norm, mixer=second.mixer, ffn=second.ffn)))
    if name == "experts":
        return changed(spec, 0, ffn=MoESpec(experts=4, top=2, expert_size=64, correction=False))
    if name == "layer norm before a feed-forward":
        return changed(spec, 0, ffn_norm=layernorm)
    if name == "layer norm before a mixer":
        return changed(spec, 1, mixer_norm=layernorm)
    if name == "no rotation":
        return changed(changed(spec, 0, mixer=replace(first.mixer, position=None)), 1, mixer=replace(second.mixer, position=None))
    if name == "part of a head":
        part = RotarySpec(theta=1e4, rotary_dim=8)
        return changed(changed(spec, 0, mixer=replace(first.mixer, position=part)), 1, mixer=replace(second.mixer, position=part))
    if name == "no feed-forward":
        return changed(spec, 0, ffn=None, ffn_norm=None)
    if name == "odd features":
        odd = SwiGLUSpec(intermediate_size=84)
        return changed(changed(spec, 0, ffn=odd), 1, ffn=odd)
    if name == "limits":
        bounded = SwiGLUSpec(intermediate_size=88, activation="quick_gelu", limit=0.7, up_shift=1.0)
        return changed(changed(spec, 0, ffn=bounded), 1, ffn=bounded)
    if name == "output bias":
        return changed(changed(spec, 0, mixer=replace(first.mixer, out_bias=True)), 1, mixer=replace(second.mixer, out_bias=True))
    if name == "one block twice":
        return replace(spec, schedule=(ScheduleEntry(0), ScheduleEntry(1), ScheduleEntry(1)))
    assert name == "two layers"
    return spec


def run(spec, weights, ids, monkeypatch, few=True, dtype=torch.bfloat16):
    from shrike_amd.kernels import ops

    calls = dict.fromkeys(NAMES, 0)

    def counted(name, fn):
        def call(*args, **kwargs):
            calls[name] += 1
            return fn(*args, **kwargs)
        return call

    with monkeypatch.context() as patch:
        for name in NAMES:
            patch.setattr(ops, name, counted(name, getattr(ops, name)))
        if not few:
            patch.setattr(ops, "few_stream_sums", lambda *sizes: 0)
            patch.setattr(ops, "few_heads_takes", lambda *sizes: False)
        runner, _, cache = make_runner(spec, weights, dtype)
        runner.use_graphs = runner.use_call_lists = False
        logits = step_whole(runner, cache, ids)
    return logits, tuple(calls.values())


@pytest.mark.parametrize("name, launches", [
    ("two layers", (3, 2, 2)), ("limits", (3, 2, 2)), ("output bias", (3, 2, 2)), ("one block twice", (5, 3, 3)),
    ("scaled residual", (0, 0, 2)), ("embedding again", (2, 2, 2)), ("vector", (2, 2, 2)), ("average", (2, 2, 2)), ("parallel block", (1, 1, 2)),
    ("experts", (1, 1, 2)), ("layer norm before a feed-forward", (2, 1, 2)), ("layer norm before a mixer", (2, 2, 2)),
    ("no rotation", (2, 2, 0)), ("part of a head", (2, 2, 0)), ("no feed-forward", (2, 1, 2)), ("odd features", (2, 2, 2))])
@pytest.mark.parametrize("n", [1, 16, 17, 64])
def test_the_launches_of_a_step_and_its_logits(name, launches, n, monkeypatch):
    spec = case(name)
    weights, ids = cpu_weights(spec), [(11 * i + 5) % 97 for i in range(n)]
    got, calls = run(spec, weights, ids, monkeypatch)
    assert calls == launches
    want, none = run(spec, weights, ids, monkeypatch, few=False)
    assert none == (0, 0, 0)
    # some twenty roundings to bfloat16 a path on either side, of 2^-9 at random: sqrt(40) * 2^-9
    assert float((got - want).norm() / want.norm()) <= 0.0125


@pytest.mark.parametrize("n, launches", [(65, (0, 0, 2)), (512, (0, 0, 2)), (513, (0, 0, 0))])
def test_longer_steps(n, launches, monkeypatch):
    spec = small_spec()
    _, model, cache = make_runner(spec, cpu_weights(spec), torch.bfloat16, num_pages=80)
    calls, ids = [0] * len(NAMES), [(11 * i + 5) % 97 for i in range(n)]
    from shrike_amd.engine.runner import ModelRunner
    from shrike_amd.engine.runtime import Runtime
    from shrike_amd.kernels import ops

    for i, name in enumerate(NAMES):
        def call(*args, i=i, fn=getattr(ops, name), **kwargs):
            calls[i] += 1
            return fn(*args, **kwargs)
        monkeypatch.setattr(ops, name, call)
    runner = ModelRunner(model, cache, Runtime("cuda:0", torch.bfloat16), graphs=False)
    step_whole(runner, cache, ids)
    assert tuple(calls) == launches


def test_float32_takes_none(monkeypatch):
    spec = small_spec()
    _, calls = run(spec, cpu_weights(spec), [1, 2, 3], monkeypatch, dtype=torch.float32)
    assert calls == (0, 0, 0)
