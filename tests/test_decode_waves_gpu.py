"""Decode attention with eight wavefronts a workgroup: contexts that give some wavefronts no chunk, one, and
several, whole and in splits, against float64; and the rule that chooses."""

import pytest
import torch


def test_the_rule():
    from shrike_amd.parts import attention
    from shrike_amd.parts.attention import decode_shares, decode_splits

    assert attention.compute_units() >= 64
    assert decode_shares(1, 2, 64, 200) == (1, 4)
    assert decode_shares(1, 2, 64, 333) == (1, 8)
    assert decode_shares(1, 2, 64, 513) == (decode_splits(1, 2, 513), 4)
    assert decode_shares(1, 2, 128, 333) == (decode_splits(1, 2, 333), 4)
    assert decode_shares(256, 2, 64, 333) == (1, 4)
    for n, ctx in ((3, 2000), (8, 2060), (40, 700), (5, 300)):  # a captured step stands for every batch and context up to its own
        assert decode_shares(n, 2, 64, ctx) == decode_shares(attention._pow2(n), 2, 64, attention._pow2(ctx))


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv_heads, head_dim, page_size, window", [(14, 2, 64, 16, None), (28, 4, 64, 16, 300),
                                                                         (3, 3, 32, 32, None), (16, 1, 64, 64, None)])
@pytest.mark.parametrize("nsplit, streaming", [(1, False), (3, True)])
def test_against_float64(heads, kv_heads, head_dim, page_size, window, nsplit, streaming):
    from shrike_amd.kernels import ops
    from tests.test_kernels_gpu import close, dev, paged_setup, put_key, reference_attention

    torch.manual_seed(heads)
    ctx = [1, 31, 33, 255, 256, 257, 513, 900]
    n, dtype = len(ctx), torch.bfloat16
    num_pages = 2 * sum(-(-c // page_size) for c in ctx) + 3
    tables, k_pool, v_pool = paged_setup(ctx, page_size, num_pages, kv_heads, head_dim, dtype, seed=1)
    for s, c in enumerate(ctx):
        for p in range(c):
            page = int(tables[s, p // page_size])
            put_key(k_pool, page, p % page_size, torch.randn(kv_heads, head_dim).to(dtype))
            v_pool[page, :, :, p % page_size] = torch.randn(kv_heads, head_dim).to(dtype)
    q = torch.randn(n, heads, head_dim).to(dtype)
    positions = torch.tensor([c - 1 for c in ctx], dtype=torch.int32)
    scale = 0.7 * head_dim**-0.5
    out = torch.empty(n, heads * head_dim, device="cuda", dtype=dtype)
    partial = torch.full((n * heads * nsplit * (head_dim + 2),), float("nan"), device="cuda")
    ops.attention_decode(dev(q).view(n, -1), out, n, heads, kv_heads, head_dim, dev(positions), tables, k_pool, v_pool, page_size,
                         window, scale, partial, nsplit, streaming, waves=8)
    want = reference_attention(q.double(), k_pool, v_pool, tables, [1] * n, [c - 1 for c in ctx], page_size, window, scale)
    assert not torch.isnan(out.float()).any(), "a slot outside the context was read"
    close(out.view(n, heads, head_dim), want, dtype, scale=1.0)
