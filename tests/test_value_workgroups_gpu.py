"""Values of 65 tokens and more on both sides of the line where their workgroups have one wavefront: each in its slot, nothing else."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_heads, head_dim", [(2, 64), (4, 128), (8, 128), (9, 128), (3, 80)])
@pytest.mark.parametrize("n", [65, 256, 257, 513, 1032])
@pytest.mark.parametrize("single", [False, True])
def test_values_reach_their_slots(kv_heads, head_dim, n, single):
    from shrike_amd.kernels import ops

    generator = torch.Generator().manual_seed(n + kv_heads)
    page, heads = 16, kv_heads
    width, seqs, longest = 3 * kv_heads * head_dim, n if single else 1, 2 if single else -(-(n + 5) // 16)
    positions = torch.arange(n) * 7 % 32 if single else torch.arange(5, 5 + n)
    token_seq = torch.arange(n) if single else torch.zeros(n, dtype=torch.long)
    tables = torch.randperm(seqs * longest, generator=generator).view(seqs, longest)
    qkv = torch.randn(n, width, generator=generator).bfloat16()
    k_pool = torch.zeros(ops.key_pool_shape(seqs * longest, kv_heads, page, head_dim), dtype=torch.bfloat16, device="cuda")
    v_pool = torch.full((seqs * longest, kv_heads, head_dim, page), float("nan"), dtype=torch.bfloat16, device="cuda")
    inv_freq = (1.0 / 1e4 ** (torch.arange(0, head_dim, 2).float() / head_dim)).cuda()
    ops.rope_kv_store(qkv.cuda(), heads, kv_heads, head_dim, head_dim, inv_freq, positions.int().cuda(), token_seq.int().cuda(),
                      tables.int().cuda(), k_pool, v_pool, page)
    expected = torch.full(v_pool.shape, float("nan"), dtype=torch.bfloat16)
    expected[tables[token_seq, positions // page], :, :, positions % page] = qkv[:, 2 * kv_heads * head_dim :].view(n, kv_heads, head_dim)
    assert torch.equal(v_pool.cpu().view(torch.int16), expected.view(torch.int16))
