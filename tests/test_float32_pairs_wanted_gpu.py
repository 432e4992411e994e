"""float32 attention with and without pairs of tokens, as the caller wants it: the same bits."""

import pytest
import torch

from tests.test_float32_attention_pairs_gpu import PAGE, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, kv_heads, head_dim", [(28, 4, 64), (64, 32, 128), (28, 14, 112), (24, 12, 256)])
@pytest.mark.parametrize("lengths", [[(0, 101)], [(250, 81), (7, 1), (8, 2), (501, 17)]])
@pytest.mark.parametrize("options", [{"window": 0}, {"window": 19}, {"window": 0, "chunk": 24, "softcap": 5.0}])
@pytest.mark.parametrize("turned", [False, True])  # (neighbours whose second token has fewer keys)
def test_the_same_bits(heads, kv_heads, head_dim, lengths, options, turned):
    from shrike_amd.kernels import ops

    positions, token_seq, tables, k_pool, v_pool = setup(lengths, kv_heads, head_dim, 600)
    if turned:
        positions, token_seq = positions.flip(0).contiguous(), token_seq.flip(0).contiguous()
    n = positions.shape[0]
    q, sinks, outs = torch.randn(n, heads * head_dim, device="cuda"), torch.randn(heads, device="cuda"), []
    for pairs in (False, True, None):
        out = torch.full((n, heads * head_dim), float("nan"), device="cuda")
        ops.attention(q, out, heads, kv_heads, head_dim, positions, token_seq, tables, k_pool, v_pool, PAGE, scale=head_dim**-0.5,
                      sinks=sinks, pairs=pairs, **options)
        outs.append(out)
    assert bool(outs[0].isfinite().all()) and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
