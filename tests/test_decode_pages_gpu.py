"""Decode attention over pages of 16, which has instances of its own, and over pages of 32 and 48: the same bits, and slots outside the
contexts, which hold NaN, are not read."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, kv_heads, head_dim, window, waves", [(14, 2, 64, None, 8), (14, 2, 64, 40, 4), (28, 4, 128, None, 4),
                                                                      (3, 1, 32, 33, 8), (5, 5, 96, None, 4), (7, 1, 256, 100, 4)])
@pytest.mark.parametrize("nsplit, streaming", [(1, True), (3, False)])
def test_pages_of_any_size_give_the_same_bits(heads, kv_heads, head_dim, window, waves, nsplit, streaming):
    from shrike_amd.kernels import ops
    from tests.test_kernels_gpu import dev, paged_setup, put_key

    ctx = [1, 16, 17, 32, 33, 47, 48, 49, 129, 400]
    n, dtype = len(ctx), torch.bfloat16
    gen = torch.Generator().manual_seed(heads)
    keys = [torch.randn(c, kv_heads, head_dim, generator=gen).to(dtype) for c in ctx]
    values = [torch.randn(c, kv_heads, head_dim, generator=gen).to(dtype) for c in ctx]
    q = torch.randn(n, heads * head_dim, generator=gen).to(dtype)
    outs = []
    for page_size in (16, 32, 48):
        tables, k_pool, v_pool = paged_setup(ctx, page_size, sum(-(-c // page_size) for c in ctx) + 2, kv_heads, head_dim, dtype, seed=3)
        for s, c in enumerate(ctx):
            for p in range(c):
                page = int(tables[s, p // page_size])
                put_key(k_pool, page, p % page_size, keys[s][p])
                v_pool[page, :, :, p % page_size] = values[s][p]
        out = torch.full((n, heads * head_dim), float("nan"), device="cuda", dtype=dtype)
        partial = torch.full((n * heads * nsplit * (head_dim + 2),), float("nan"), device="cuda")
        ops.attention_decode(dev(q), out, n, heads, kv_heads, head_dim, dev(torch.tensor(ctx, dtype=torch.int32) - 1), tables, k_pool,
                             v_pool, page_size, window, head_dim**-0.5, partial, nsplit, streaming, waves=waves)
        outs.append(out)
    assert bool(outs[0].float().isfinite().all()) and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
