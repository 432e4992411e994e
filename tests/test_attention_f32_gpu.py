"""Float32 attention on the matrix units at the edges of its blocks of 256 keys: against float64, and the
same bits whether a token's blocks are formed by one workgroup or by several."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

POSITIONS = [0, 1, 15, 63, 64, 254, 255, 256, 257, 511, 700]


@pytest.mark.parametrize("heads, kv_heads, head_dim, v_dim, page, window, chunk, extras", [
    (14, 2, 64, 64, 16, None, None, False),
    (3, 3, 20, 20, 4, None, None, True),
    (20, 1, 96, 36, 8, 300, None, True),
    (40, 2, 256, 256, 64, None, None, False),
    (6, 2, 32, 130, 16, 257, None, False),
    (4, 4, 128, 128, 32, None, 256, True),
])
def test_edges_of_the_blocks(heads, kv_heads, head_dim, v_dim, page, window, chunk, extras):
    from shrike_amd.kernels import ops

    torch.manual_seed(heads + head_dim)
    n, per, ctx = len(POSITIONS), -(-704 // page), 704
    num_pages = n * per + 2
    slab = ops.key_slab(head_dim)
    k_pool = torch.full((num_pages, kv_heads, head_dim // slab, page, slab), float("nan"), device="cuda")
    v_pool = torch.full((num_pages, kv_heads, v_dim, page), float("nan"), device="cuda")
    tables = torch.randperm(num_pages - 2, device="cuda")[: n * per].view(n, per).int()
    keys, values = torch.randn(n, ctx, kv_heads, head_dim, device="cuda"), torch.randn(n, ctx, kv_heads, v_dim, device="cuda")
    for t, pos in enumerate(POSITIONS):  # what lies behind the token stays not-a-number
        at = torch.arange(pos + 1, device="cuda")
        rows = tables[t].long()[at // page]
        k_pool[rows, :, :, at % page] = keys[t, : pos + 1].view(pos + 1, kv_heads, head_dim // slab, slab)
        v_pool[rows, :, :, at % page] = values[t, : pos + 1]
    q = torch.randn(n, heads * head_dim, device="cuda")
    positions = torch.tensor(POSITIONS, dtype=torch.int32, device="cuda")
    seqs = torch.arange(n, dtype=torch.int32, device="cuda")
    scale = 1.3 / math.sqrt(head_dim)
    more = dict(softcap=6.0, sinks=torch.randn(heads, device="cuda"), dist_bias=torch.randn(heads, 19, device="cuda")) if extras else {}

    def run(rows, splits):
        out = torch.full((rows.numel(), heads * v_dim), 9.0, device="cuda")
        partial = None
        if splits > 1:
            partial = torch.full((ops.attention_partial_floats(rows.numel(), heads, v_dim, per, page),), float("nan"), device="cuda")
        ops.attention(q[rows], out, heads, kv_heads, head_dim, positions[rows], seqs[rows], tables, k_pool, v_pool, page, window,
                      scale, chunk=chunk, v_dim=v_dim, partial=partial, splits=splits, **more)
        return out

    every = torch.arange(n, device="cuda")
    whole = run(every, 1)
    for splits in (2, 3, 9):
        assert torch.equal(run(every, splits), whole)
    assert torch.equal(run(every[-2:-1], 1), whole[-2:-1])
    for t, pos in enumerate(POSITIONS):
        lo = max(0, pos - window + 1) if window else 0
        lo = max(lo, pos // chunk * chunk) if chunk else lo
        for h in range(heads):
            g = h // (heads // kv_heads)
            s = keys[t, lo : pos + 1, g].double() @ q[t, h * head_dim : (h + 1) * head_dim].double() * scale
            if extras:
                s = 6.0 * torch.tanh(s / 6.0)
                far = (pos - torch.arange(lo, pos + 1, device="cuda")).clamp(max=18)
                s = s + more["dist_bias"][h, far].double()
            with_sink = torch.cat([s, more["sinks"][h : h + 1].double()]) if extras else s
            weights = torch.exp(s - torch.logsumexp(with_sink, 0))
            want = weights @ values[t, lo : pos + 1, g].double()
            # a score of size ~10 is off by some ulp, a weight by as much relatively; the sums add half an ulp
            # of values of order one a term, a few hundred terms weighted to one
            assert torch.allclose(whole[t, h * v_dim : (h + 1) * v_dim].double(), want, atol=2e-5, rtol=0), (t, h)


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("sinks", [False, True])
def test_scores_of_minus_infinity(splits, sinks):
    """A table of distances that rules out the nearest keys, whole blocks of them, or the far ones: what is left is the
    softmax; where nothing is left, nothing beside the sink, or no number without one."""
    from shrike_amd.kernels import ops

    torch.manual_seed(3)
    heads, dim, page, ctx = 4, 32, 16, 1024
    k_pool = torch.randn(ctx // page, 1, dim // ops.key_slab(dim), page, ops.key_slab(dim), device="cuda")
    v_pool = torch.randn(ctx // page, 1, dim, page, device="cuda")
    tables = torch.arange(ctx // page, device="cuda").int().view(1, -1)
    keys = k_pool.permute(0, 3, 1, 2, 4).reshape(ctx, dim)
    values = v_pool.permute(0, 3, 1, 2).reshape(ctx, dim)
    positions = torch.tensor([5, 255, 256, 700, 1023], dtype=torch.int32, device="cuda")
    n = positions.numel()
    q = torch.randn(n, heads * dim, device="cuda")
    bias = torch.randn(heads, 1024, device="cuda")
    bias[0, :300] = -float("inf")  # the nearest block and more
    bias[1, 10:] = -float("inf")  # all but the nearest ten: whole blocks in front
    bias[2, 100:900] = -float("inf")
    sink = torch.randn(heads, device="cuda") if sinks else None
    out = torch.full((n, heads * dim), 9.0, device="cuda")
    partial = torch.full((ops.attention_partial_floats(n, heads, dim, ctx // page, page),), float("nan"), device="cuda")
    ops.attention(q, out, heads, 1, dim, positions, torch.zeros(n, dtype=torch.int32, device="cuda"), tables, k_pool, v_pool, page, None,
                  dim**-0.5, dist_bias=bias, sinks=sink, **(dict(partial=partial, splits=splits) if splits > 1 else {}))
    got = out.view(n, heads, dim).double()
    for t, pos in enumerate(positions.tolist()):
        for h in range(heads):
            s = keys[: pos + 1].double() @ q[t, h * dim : (h + 1) * dim].double() * dim**-0.5
            s = s + bias[h, pos - torch.arange(pos + 1, device="cuda")].double()
            top = torch.cat([s, sink[h : h + 1].double()]) if sinks else s
            if bool(torch.isinf(top).all()):
                assert bool(torch.isnan(got[t, h]).all())
                continue
            want = torch.exp(s - torch.logsumexp(top, 0)) @ values[: pos + 1].double()
            assert torch.allclose(got[t, h], want, atol=2e-5, rtol=0), (t, h)


@pytest.mark.parametrize("heads, kv_heads, dim, page, window", [(4, 1, 32, 16, None), (4, 2, 40, 4, None), (14, 2, 64, 16, 20), (5, 5, 48, 8, 33),
                                                              (3, 1, 80, 16, None), (6, 2, 132, 16, 17)])
def test_steps_without_a_key_that_is_read(heads, kv_heads, dim, page, window):
    """Prompts of up to 100 tokens: every number of steps of 16 keys, and of pairs of them, that hold one."""
    from shrike_amd.kernels import ops

    torch.manual_seed(dim)
    n, slab = 100, ops.key_slab(dim)
    pages = -(-n // page)
    k_pool = torch.full((pages + 1, kv_heads, dim // slab, page, slab), float("nan"), device="cuda")
    v_pool = torch.full((pages + 1, kv_heads, dim, page), float("nan"), device="cuda")
    tables = torch.randperm(pages + 1, device="cuda")[:pages].int().view(1, -1)
    keys, values = torch.randn(n, kv_heads, dim, device="cuda"), torch.randn(n, kv_heads, dim, device="cuda")
    at = torch.arange(n, device="cuda")
    k_pool[tables[0].long()[at // page], :, :, at % page] = keys.view(n, kv_heads, dim // slab, slab)
    v_pool[tables[0].long()[at // page], :, :, at % page] = values
    q, out = torch.randn(n, heads * dim, device="cuda"), torch.empty(n, heads * dim, device="cuda")
    ops.attention(q, out, heads, kv_heads, dim, at.int(), torch.zeros(n, dtype=torch.int32, device="cuda"), tables, k_pool, v_pool, page,
                  window, dim**-0.5)
    s = torch.einsum("thd,khd->htk", q.view(n, heads, dim).double(), keys.repeat_interleave(heads // kv_heads, 1).double()) * dim**-0.5
    far = at.view(-1, 1) - at
    s = s.masked_fill((far < 0) | (far >= (window or n)), -float("inf"))
    want = torch.einsum("htk,khd->thd", torch.softmax(s, -1), values.repeat_interleave(heads // kv_heads, 1).double())
    # (scores of a few units off by some ulp, weights by as much; half an ulp of values of order one a term)
    assert torch.allclose(out.view(n, heads, dim).double(), want, atol=1e-5, rtol=0)
