"""Among how many workgroups a step of single tokens shares their rows in latent attention: in the portions' kernel shares of 64 rows as long as
there is a compute unit for each, in the kernel for single tokens shares of 128; alike for every number of tokens up to a power of two (CPU)."""

import numpy as np
import pytest

from shrike_amd.config.specs import LatentAttentionSpec
from shrike_amd.engine.context import StepShape
from shrike_amd.kernels import ops
from shrike_amd.parts import latent_attention
from shrike_amd.parts.base import build_part


def plan(monkeypatch, contexts, portion=None, latent=448, heads=28, window=None):
    monkeypatch.setattr(latent_attention, "compute_units", lambda: 256)
    spec = LatentAttentionSpec(num_heads=heads, head_dim=128, rot_dim=64, value_dim=128, q_rank=64, kv_rank=latent, scale=0.1, eps=1e-5,
                               rot_theta=1e4, window=window)
    mixer = build_part("mixer", spec, 256, "m")
    mixer.mfma = True
    mixer.prompt_tokens = ops.latent_prompt_tokens(heads, latent + 64, latent)
    lengths = [1] * len(contexts) + ([] if portion is None else [portion])
    shape = StepShape(np.array(lengths), np.array([c - 1 for c in contexts] + ([] if portion is None else [0])), 16)
    mixer.prepare(shape)
    (nsplit, group, first, prompt_split, tokens), = shape.notes.values()
    return nsplit, group, first


@pytest.mark.parametrize("contexts, nsplit", [
    ([60], 1), ([65], 2), ([850], 16), ([850] * 8, 16), ([850] * 5 + [60] * 3, 16), ([1500] * 16, 16), ([1500] * 9, 16), ([1500] * 32, 16),
    ([1500] * 64, 8), ([5000], 64), ([20000], 64), ([20000] * 256, 2), ([20000] * 512, 1)])
def test_shares_of_single_tokens(contexts, nsplit, monkeypatch):
    assert plan(monkeypatch, contexts) == (nsplit, 1, len(contexts))


def test_a_window_bounds_them(monkeypatch):
    assert plan(monkeypatch, [20000], window=100) == (2, 1, 1)


def test_the_kernel_for_single_tokens_has_shares_of_128(monkeypatch):
    assert plan(monkeypatch, [850] * 8, latent=56, heads=8) == (8, 1, 8)


def test_single_tokens_beside_a_portion(monkeypatch):
    assert plan(monkeypatch, [850] * 8, portion=40) == (8, 1, 8)
