"""float32 attention with and without pairs of tokens, as the caller wants it: the same bits."""

import pytest
import torch

from tests.test_float32_attention_pairs_gpu import PAGE, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, kv_heads, head_dim", [(28, 4, 64), (64, 32, 128), (28, 14, 112), (24, 12, 256)])
@pytest.mark.parametrize("lengths", [[(0, 101)], [(250, 81), (7, 1), (8, 2), (501, 17)]])
def test_the_same_bits(heads, kv_heads, head_dim, lengths):
    from shrike_amd.kernels import ops

    positions, token_seq, tables, k_pool, v_pool = setup(lengths, kv_heads, head_dim, 600)
    n = positions.shape[0]
    q, outs = torch.randn(n, heads * head_dim, device="cuda"), []
    for pairs in (False, True, None):
        out = torch.full((n, heads * head_dim), float("nan"), device="cuda")
        ops.attention(q, out, heads, kv_heads, head_dim, positions, token_seq, tables, k_pool, v_pool, PAGE, scale=head_dim**-0.5,
                      window=0, pairs=pairs)
        outs.append(out)
    assert bool(outs[0].isfinite().all()) and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
