"""Values of 65 tokens and more go to their pages eight neighbouring tokens at a time: in one piece where they lie side by side there,
one by one elsewhere (portions that begin inside a piece, sequences that end inside a group, pages of other sizes, remainders)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits", [0, 1, 3])
@pytest.mark.parametrize("portions", [[(0, 65)], [(0, 72)], [(16, 80), (3, 29)], [(8, 24), (0, 41), (40, 7)], [(13, 131)]])
@pytest.mark.parametrize("kv_heads, head_dim, page_size", [(2, 64, 16), (3, 96, 8), (1, 32, 12), (4, 128, 24)])
def test_values_reach_their_slots_and_nothing_else(kv_heads, head_dim, page_size, portions, splits):
    from shrike_amd.kernels import ops

    generator = torch.Generator().manual_seed(len(portions) + splits)
    heads, n = 2 * kv_heads, sum(count for _, count in portions)
    width = (heads + 2 * kv_heads) * head_dim
    positions = torch.cat([torch.arange(start, start + count) for start, count in portions]).int()
    token_seq = torch.cat([torch.full((count,), i) for i, (_, count) in enumerate(portions)]).int()
    longest = max(-(-(start + count) // page_size) for start, count in portions)
    pages = longest * len(portions) + 3
    tables = torch.randperm(pages, generator=generator)[: longest * len(portions)].int().view(len(portions), longest)
    slab = ops.key_slab(head_dim)
    k_pool = torch.zeros(pages, kv_heads, head_dim // slab, page_size, slab, dtype=torch.bfloat16, device="cuda")
    v_pool = torch.full((pages, kv_heads, head_dim, page_size), float("nan"), dtype=torch.bfloat16, device="cuda")
    qkv = torch.randn(n, width, generator=generator).bfloat16()
    split_sum, values = None, qkv
    if splits:
        parts, bias = torch.randn(splits, n, width, generator=generator), torch.randn(width, generator=generator)
        split_sum = ops.SplitSum(parts.cuda(), bias.cuda())
        values = parts[0]
        for z in range(1, splits):
            values = values + parts[z]
        values = (values + bias).bfloat16()  # (the same additions in the same order: the same bits)
    inv_freq = (1.0 / 1e4 ** (torch.arange(0, head_dim, 2).float() / head_dim)).cuda()
    ops.rope_kv_store(qkv.cuda(), heads, kv_heads, head_dim, head_dim, inv_freq, positions.cuda(), token_seq.cuda(), tables.cuda(),
                      k_pool, v_pool, page_size, split_sum=split_sum)
    expected = torch.full(v_pool.shape, float("nan"), dtype=torch.bfloat16)
    values = values[:, (heads + kv_heads) * head_dim :].view(n, kv_heads, head_dim)
    for t in range(n):
        pos = int(positions[t])
        expected[int(tables[int(token_seq[t]), pos // page_size]), :, :, pos % page_size] = values[t]
    assert torch.equal(v_pool.cpu().view(torch.int16), expected.view(torch.int16))
