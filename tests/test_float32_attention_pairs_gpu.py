"""float32 attention whose workgroups take two neighbouring tokens of a sequence: the bits of every token by itself."""

import pytest
import torch

pytestmark = pytest.mark.gpu

PAGE = 16


def setup(lengths, kv_heads, head_dim, width):
    from shrike_amd.kernels import ops

    torch.manual_seed(len(lengths) + head_dim)
    blocks = -(-width // PAGE)
    pages = blocks * len(lengths)
    tables = torch.randperm(pages, device="cuda").to(torch.int32).view(len(lengths), blocks)
    k_pool = torch.randn(ops.key_pool_shape(pages, kv_heads, PAGE, head_dim), device="cuda")
    v_pool = torch.randn(pages, kv_heads, head_dim, PAGE, device="cuda")
    positions = torch.cat([torch.arange(first, first + n) for first, n in lengths]).to(torch.int32).cuda()
    token_seq = torch.cat([torch.full((n,), i) for i, (_, n) in enumerate(lengths)]).to(torch.int32).cuda()
    return positions, token_seq, tables, k_pool, v_pool


@pytest.mark.parametrize("heads, kv_heads, head_dim", [(28, 4, 64), (24, 24, 32), (32, 8, 48), (64, 32, 128), (12, 12, 96)])
@pytest.mark.parametrize("lengths", [[(0, 101)], [(250, 81), (7, 1), (8, 2), (501, 17)], [(240, 97)]])
@pytest.mark.parametrize("options", [{"window": 0}, {"window": 19}, {"window": 0, "chunk": 24, "softcap": 5.0}])
def test_the_same_bits_as_one_token_at_a_time(heads, kv_heads, head_dim, lengths, options):
    from shrike_amd.kernels import ops

    positions, token_seq, tables, k_pool, v_pool = setup(lengths, kv_heads, head_dim, 600)
    n = positions.shape[0]
    q, sinks = torch.randn(n, heads * head_dim, device="cuda"), torch.randn(heads, device="cuda")

    def run(rows):
        out = torch.empty(len(rows), heads * head_dim, device="cuda")
        ops.attention(q[rows].contiguous(), out, heads, kv_heads, head_dim, positions[rows].contiguous(), token_seq[rows].contiguous(),
                      tables, k_pool, v_pool, PAGE, scale=head_dim**-0.5, sinks=sinks, **options)
        return out

    want = torch.cat([run([t]) for t in range(n)])
    assert bool(want.isfinite().all()) and torch.equal(run(list(range(n))), want)
    turned = list(range(n))[::-1]  # neighbours whose second token has fewer keys
    assert torch.equal(run(turned), want[turned])


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_token_does_not_meet_values_that_only_its_neighbour_reads(bad):
    from shrike_amd.kernels import ops

    heads, kv_heads, head_dim = 24, 12, 64  # (480 workgroups by token: in pairs)
    positions, token_seq, tables, k_pool, v_pool = setup([(0, 40)], kv_heads, head_dim, 64)
    q, window = torch.randn(40, heads * head_dim, device="cuda"), 8
    for at in (16, 17):  # the second of one pair of tokens, the first of another
        values = v_pool.clone()
        values[tables[0, at // PAGE].long(), :, :, at % PAGE] = bad
        got, want = (torch.empty(40, heads * head_dim, device="cuda") for _ in range(2))
        for v, out in ((values, got), (v_pool, want)):
            ops.attention(q, out, heads, kv_heads, head_dim, positions, token_seq, tables, k_pool, v, PAGE, scale=0.125, window=window)
        apart = [t for t in range(40) if not at <= t < at + window]
        assert torch.equal(got[apart], want[apart])
        assert not bool(got[at : at + window].isfinite().any())
