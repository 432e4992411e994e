"""Rotation and cache write in vectors where queries and keys alone fill a workgroup's items: against the general kernel, which takes rows
that are not aligned."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, kv_heads, head_dim", [(64, 64, 128), (120, 8, 128), (112, 16, 128), (121, 8, 128), (96, 32, 64), (32, 32, 256)])
@pytest.mark.parametrize("n", [65, 128, 130])
def test_vectors_and_elements_agree(heads, kv_heads, head_dim, n):
    from shrike_amd.kernels import ops

    torch.manual_seed(heads + n)
    page, width = 16, (heads + 2 * kv_heads) * head_dim
    pages = -(-(n + 3) // page)
    tables = torch.randperm(pages).int().view(1, pages).cuda()
    positions, token_seq = torch.arange(3, 3 + n).int().cuda(), torch.zeros(n, dtype=torch.int32, device="cuda")
    inv_freq = (1.0 / 1e4 ** (torch.arange(0, head_dim, 2).float() / head_dim)).cuda()
    rows, results = torch.randn(n, width).bfloat16(), []
    for shift in (0, 1):
        room = torch.zeros(n * width + 1, dtype=torch.bfloat16, device="cuda")
        qkv = room[shift : shift + n * width].view(n, width)
        qkv.copy_(rows)
        k_pool = torch.zeros(ops.key_pool_shape(pages, kv_heads, page, head_dim), dtype=torch.bfloat16, device="cuda")
        v_pool = torch.zeros(pages, kv_heads, head_dim, page, dtype=torch.bfloat16, device="cuda")
        ops.rope_kv_store(qkv, heads, kv_heads, head_dim, head_dim, inv_freq, positions, token_seq, tables, k_pool, v_pool, page)
        results.append((qkv[:, : heads * head_dim].clone(), k_pool, v_pool))
    for vectors, elements in zip(*results):
        assert torch.equal(vectors.view(torch.int16), elements.view(torch.int16))
