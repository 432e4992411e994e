"""Prompt attention with 32 rows a wavefront: every size of group, head and page, edges of chunks, shares of keys."""

import pytest
import torch

from tests.test_kernels_gpu import close, dev, fill_pools, paged_setup, reference_attention

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from shrike_amd.kernels import ops

    return ops


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


def run(ops, heads, kv_heads, head_dim, page_size, window, chunk, nsplit, singles, seq_lens, starts, sinks=None):
    """(out, reference) of a step whose first `singles` sequences are single tokens."""
    torch.manual_seed(20)
    dtype = torch.bfloat16
    queries = ops.attention_prefill_rows_queries(heads, kv_heads, head_dim)
    assert queries == 256 // (heads // kv_heads)
    ctx = [s + n for s, n in zip(starts, seq_lens)]
    n = sum(seq_lens)
    num_pages = sum(-(-c // page_size) for c in ctx) + 5
    tables, k_pool, v_pool = paged_setup(ctx, page_size, num_pages, kv_heads, head_dim, dtype, seed=5)
    fill_pools(tables, k_pool, v_pool, ctx, page_size)
    q = torch.randn(n, heads, head_dim).to(dtype)
    cu = [0]
    for length in seq_lens:
        cu.append(cu[-1] + length)
    entries = [(s, q0) for s, length in enumerate(seq_lens) if s >= singles for q0 in range(0, length, queries)]
    entries.reverse()
    out = torch.full((n, heads * head_dim), float("nan"), device="cuda", dtype=dtype)
    partial = torch.full(((n - singles) * heads * nsplit * (head_dim + 2),), float("nan"), device="cuda")
    ops.attention_prefill_shared(dev(q).view(n, -1), out, len(entries), heads, kv_heads, head_dim, i32(cu), i32(ctx),
                                 i32([e[0] for e in entries]), i32([e[1] for e in entries]), tables, k_pool, v_pool, page_size,
                                 window, head_dim**-0.5, small=2, partial=partial, nsplit=nsplit, first_token=singles, chunk=chunk,
                                 sinks=sinks)
    assert torch.isnan(out[:singles].float()).all() and not torch.isnan(out[singles:].float()).any()
    got = out[singles:].view(n - singles, heads, head_dim)
    return got, (q, k_pool, v_pool, tables)


@pytest.mark.parametrize("heads, kv_heads, head_dim, page_size, window",
                         [(14, 2, 64, 16, None), (28, 4, 128, 16, None), (40, 8, 128, 16, 100), (16, 2, 64, 48, 17), (12, 1, 128, 32, 50),
                          (34, 2, 64, 16, None), (8, 2, 128, 64, None), (4, 1, 64, 80, 64)])
@pytest.mark.parametrize("nsplit, singles", [(1, 0), (3, 5), (8, 0)])
def test_rows_against_the_reference(ops, heads, kv_heads, head_dim, page_size, window, nsplit, singles):
    seq_lens = [1] * singles + [2, 200, 16, 64, 37, 130, 65, 1]
    starts = [9, 40, 0, 77, 16][:singles] + [0, 60, 5, 0, 91, 31, 63, 127]
    got, (q, k_pool, v_pool, tables) = run(ops, heads, kv_heads, head_dim, page_size, window, None, nsplit, singles, seq_lens, starts)
    want = reference_attention(q.double(), k_pool, v_pool, tables, seq_lens, starts, page_size, window, head_dim**-0.5)
    close(got, want[singles:], torch.bfloat16, scale=1.0)


def test_a_block_local_mask_and_many_chunks(ops):
    """Blocks of 96 keys that end inside chunks of 64; 700 keys before the portion."""
    seq_lens, starts = [150, 33], [700, 5]
    got, (q, k_pool, v_pool, tables) = run(ops, 28, 4, 128, 16, None, 96, 1, 0, seq_lens, starts)
    for i, (s, row) in enumerate((s, r) for s in range(2) for r in range(seq_lens[s])):
        pos = starts[s] + row
        lo = pos // 96 * 96
        want = reference_attention(q[i : i + 1].double(), k_pool, v_pool, tables[s : s + 1], [1], [pos], 16, pos - lo + 1, 128**-0.5)
        close(got[i : i + 1], want, torch.bfloat16, scale=1.0)


def test_sinks_join_the_sum(ops):
    """A sink is one more term of a head's denominator, with one workgroup an entry and with shares."""
    heads, kv_heads, d = 14, 2, 64
    sinks = torch.randn(heads, device="cuda")
    seq_lens, starts = [100, 40], [300, 0]
    outs = [run(ops, heads, kv_heads, d, 16, None, None, nsplit, 0, seq_lens, starts, sinks=sinks)[0] for nsplit in (1, 4)]
    plain, (q, k_pool, v_pool, tables) = run(ops, heads, kv_heads, d, 16, None, None, 1, 0, seq_lens, starts)
    # the denominators, from the scores in double precision
    at = 0
    for s, (length, start) in enumerate(zip(seq_lens, starts)):
        keys = torch.stack([torch.stack([k_pool[int(tables[s, p // 16]), g].transpose(0, 1).reshape(16, d)[p % 16] for p in range(start + length)])
                            for g in range(kv_heads)]).double()
        for i in range(0, length, 13):
            for h in range(heads):
                score = (keys[h // 7, : start + i + 1] @ dev(q[at + i, h]).double()) * d**-0.5
                share = score.exp().sum() / (score.exp().sum() + sinks[h].double().exp())
                for out in outs:
                    close(out[at + i, h].double(), (plain[at + i, h].double() * share).cpu(), torch.bfloat16, scale=1.0)
        at += length


@pytest.mark.parametrize("heads, kv_heads, head_dim, nsplit, at", [(14, 2, 64, 1, 3), (28, 4, 128, 1, 31), (28, 4, 128, 3, 200), (28, 4, 128, 1, 400)])
def test_an_infinite_value_is_an_infinite_result_and_no_other(ops, heads, kv_heads, head_dim, nsplit, at, monkeypatch):
    """One element of the value of a key that every query reads is infinity, in the first tile that a workgroup reads or a
    later one: each gets infinity for that element, and nothing else changes."""
    import sys

    element, page_size, seq_lens, starts = 5, 16, [30], [500]
    plain, _ = run(ops, heads, kv_heads, head_dim, page_size, None, None, nsplit, 0, seq_lens, starts)
    fill = fill_pools

    def fill_and_spoil(tables, k_pool, v_pool, ctx, page_size):
        fill(tables, k_pool, v_pool, ctx, page_size)
        v_pool[int(tables[0, at // page_size]), :, element, at % page_size] = float("inf")

    monkeypatch.setattr(sys.modules[__name__], "fill_pools", fill_and_spoil)
    got, _ = run(ops, heads, kv_heads, head_dim, page_size, None, None, nsplit, 0, seq_lens, starts)
    assert bool((got[..., element] == float("inf")).all())
    others = [e for e in range(head_dim) if e != element]
    assert torch.equal(got[..., others], plain[..., others])
