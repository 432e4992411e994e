"""Which latent attentions serve single tokens in the prompt portions' kernel: the sizes at which it is the faster one (CPU)."""

from types import SimpleNamespace

import pytest

from shrike_amd.kernels import ops
from shrike_amd.parts.latent_attention import LatentAttention


@pytest.mark.parametrize("heads, latent, rotated, alike", [
    (28, 448, 64, True), (14, 112, 32, True), (4, 80, 16, True), (3, 112, 32, False), (14, 64, 8, False), (28, 56, 8, False), (32, 160, 16, True),
    (33, 160, 16, False), (64, 160, 16, False), (65, 160, 16, True), (33, 128, 16, True), (33, 256, 8, True), (28, 512, 64, False)])
def test_by_heads_and_rows(heads, latent, rotated, alike):
    mixer = SimpleNamespace(spec=SimpleNamespace(num_heads=heads, kv_rank=latent, rot_dim=rotated),
                            prompt_tokens=ops.latent_prompt_tokens(heads, latent + rotated, latent))
    assert LatentAttention.single_in_prompt.fget(mixer) is alike
