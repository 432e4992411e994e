"""The retention scan's vector accesses, with and without a decay of its own for every key channel."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim, v_dim, heads, seqs", [(128, 256, 14, 8), (8, 5, 2, 3), (72, 16, 3, 2), (520, 4, 1, 2), (1024, 3, 1, 1)])
@pytest.mark.parametrize("gated", [True, False])
def test_a_scan_in_vectors_has_the_bits_of_one_element_by_element(dim, v_dim, heads, seqs, gated):
    from shrike_amd.kernels import ops

    torch.manual_seed(dim + v_dim)
    qk, v = heads * dim, heads * v_dim
    n = seqs + 2  # (the last sequence has three tokens)
    proj = torch.randn(n, 2 * qk + v, device="cuda").bfloat16()
    cu = torch.tensor([*range(seqs), n], dtype=torch.int32, device="cuda")
    positions = torch.tensor([5] * (seqs - 1) + [0, 1, 2], dtype=torch.int32, device="cuda")
    slots = torch.arange(seqs - 1, -1, -1, dtype=torch.int32, device="cuda")
    size = heads * v_dim * dim
    start = torch.randn(seqs, size, device="cuda")
    log_decay = -torch.rand(n, qk, device="cuda") if gated else None
    decay = None if gated else torch.rand(heads, device="cuda")
    results = []
    for stride, offset in ((-(-size // 4) * 4 + 4, 0), (size | 1, 1)):  # (the second: states that are not aligned)
        held = torch.empty(seqs * stride + 1, device="cuda")
        state = held[offset : offset + seqs * stride].view(seqs, stride)[:, :size]
        state.copy_(start)
        out = torch.empty(n, v, device="cuda")
        ops.retention_scan(proj, 0, qk, 2 * qk, decay, seqs, heads, dim, v_dim, positions, cu, slots, state, out, log_decay=log_decay,
                           q_scale=0.3)
        results.append((state.clone(), out))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
