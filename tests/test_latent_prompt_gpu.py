"""Latent attention of prompt portions: portions of several sequences whose ends fall within a workgroup's
tokens, rows and values of every size class, windows and block-local masks, rows shared among workgroups,
not-numbers wherever nothing may be read."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, key_dim, v_dim, page, window, chunk", [
    (28, 512, 448, 16, None, None), (14, 160, 128, 16, None, None), (3, 40, 24, 4, None, 64), (64, 264, 200, 32, 70, None),
    (112, 512, 500, 16, None, None), (1, 8, 3, 8, 33, None), (17, 256, 256, 64, None, None), (128, 320, 250, 16, 100, 128),
])
@pytest.mark.parametrize("nsplit", [1, 3])
def test_against_float64(heads, key_dim, v_dim, page, window, chunk, nsplit):
    from shrike_amd.kernels import ops

    assert ops.latent_prompt_tokens(heads, key_dim, v_dim) >= 1
    torch.manual_seed(heads + key_dim)
    starts, lengths = [0, 61, 0, 130], [45, 7, 1, 35]  # (one-token portions are served too)
    n, ctx = sum(lengths), [s + k for s, k in zip(starts, lengths)]
    per = -(-max(ctx) // page)
    pool = torch.full((4 * per + 1, page, key_dim), float("nan"), device="cuda", dtype=torch.bfloat16)
    tables = torch.randperm(4 * per + 1)[: 4 * per].view(4, per).int()
    rows = [torch.randn(c, key_dim).bfloat16() for c in ctx]
    for s, r in enumerate(rows):
        at = torch.arange(r.shape[0])
        pool[tables[s].long()[at // page].cuda(), (at % page).cuda()] = r.cuda()
    q = torch.randn(n, heads, key_dim).bfloat16()
    positions = torch.cat([torch.arange(s, s + k) for s, k in zip(starts, lengths)])
    seqs = torch.repeat_interleave(torch.arange(4), torch.tensor(lengths))
    scale = 0.7 / key_dim**0.5
    out = torch.full((n, heads * v_dim), float("nan"), device="cuda", dtype=torch.bfloat16)
    partial = torch.full((n * heads * nsplit * (v_dim + 2),), float("nan"), device="cuda")
    ops.latent_prompt(q.view(n, -1).cuda(), out, heads, key_dim, v_dim, positions.int().cuda(), seqs.int().cuda(), tables.cuda(),
                      pool, page, window, scale, chunk=chunk, partial=partial, nsplit=nsplit)
    got = out.view(n, heads, v_dim).double().cpu()
    for t in range(n):
        p = int(positions[t])
        lo = max(0, p - window + 1) if window else 0
        lo = max(lo, p // chunk * chunk) if chunk else lo
        r = rows[int(seqs[t])][lo : p + 1].double()
        w = torch.softmax(q[t].double() @ r.T * scale, -1)
        want = w @ r[:, :v_dim]
        # weights and the result are rounded to bfloat16 (2^-9 each, the weights' sizes adding up to one)
        bound = 2.0**-7 * (w @ r[:, :v_dim].abs()) + 1e-3
        assert bool(((got[t] - want).abs() <= bound).all()), t


@pytest.mark.parametrize("heads, key_dim, v_dim, window, chunk", [
    (28, 512, 448, None, None), (14, 160, 128, None, None), (3, 40, 24, None, 64), (64, 264, 200, 70, None), (1, 8, 8, 33, None),
    (17, 256, 256, None, None), (9, 320, 250, 100, 128),
])
@pytest.mark.parametrize("nsplit", [1, 3])
def test_a_row_that_is_no_number_stays_with_the_tokens_that_read_it(heads, key_dim, v_dim, window, chunk, nsplit):
    """Infinities and NaN in one sequence's rows, from some position on: tokens of other sequences in the same
    workgroups, earlier ones of the same sequence and later ones whose window has passed them keep their bits."""
    from shrike_amd.kernels import ops

    page = 16
    torch.manual_seed(heads + key_dim)
    starts, lengths = [0, 61, 0, 130, 3], [45, 7, 1, 35, 150]
    n, ctx = sum(lengths), [s + k for s, k in zip(starts, lengths)]
    per = -(-max(ctx) // page)
    tables = torch.randperm(5 * per).view(5, per).int().cuda()
    clean = torch.randn(5 * per, page, key_dim, device="cuda").bfloat16()
    q = torch.randn(n, heads * key_dim, device="cuda").bfloat16()
    positions = torch.cat([torch.arange(s, s + k) for s, k in zip(starts, lengths)]).int().cuda()
    seqs = torch.repeat_interleave(torch.arange(5), torch.tensor(lengths)).int().cuda()

    def run(pool):
        out = torch.full((n, heads * v_dim), 9.0, device="cuda", dtype=torch.bfloat16)
        partial = torch.full((n * heads * nsplit * (v_dim + 2),), float("nan"), device="cuda")
        ops.latent_prompt(q, out, heads, key_dim, v_dim, positions, seqs, tables, pool, page, window, 0.7 / key_dim**0.5,
                          chunk=chunk, partial=partial, nsplit=nsplit)
        return out

    want = run(clean)
    assert bool(torch.isfinite(want.float()).all())
    p = positions.long()
    lo = torch.zeros_like(p)
    if window:
        lo = torch.maximum(lo, p - window + 1)
    if chunk:
        lo = torch.maximum(lo, p // chunk * chunk)
    for seq, at, what in ((0, 17, float("nan")), (1, 67, float("inf")), (3, 140, float("-inf")), (4, 40, float("nan"))):
        pool = clean.clone()
        pool[tables[seq, at // page].long(), at % page, v_dim // 2] = what
        got = run(pool)
        reads = (seqs == seq) & (lo <= at) & (at <= p)
        assert bool(reads.any())
        assert torch.equal(got[~reads], want[~reads]), (seq, at)
        assert not bool(torch.isfinite(got[reads].float()).view(-1, heads, v_dim)[:, :, v_dim // 2].any()), (seq, at)


@pytest.mark.parametrize("heads, key_dim, v_dim, window", [(28, 512, 448, None), (14, 160, 128, 70), (1, 64, 62, None), (8, 320, 256, None)])
def test_any_number_of_tokens_a_workgroup(heads, key_dim, v_dim, window):
    """The same bits with one token a workgroup, a few, and as many as fit; results at any address."""
    from shrike_amd.kernels import KernelError, ops

    page, most = 16, ops.latent_prompt_tokens(heads, key_dim, v_dim)
    torch.manual_seed(heads)
    starts, lengths = [0, 61, 200, 0], [45, 7, 130, 2]
    n, ctx = sum(lengths), [s + k for s, k in zip(starts, lengths)]
    per = -(-max(ctx) // page)
    tables = torch.randperm(4 * per).view(4, per).int().cuda()
    pool = torch.randn(4 * per, page, key_dim, device="cuda").bfloat16()
    q = torch.randn(n, heads * key_dim, device="cuda").bfloat16()
    positions = torch.cat([torch.arange(s, s + k) for s, k in zip(starts, lengths)]).int().cuda()
    seqs = torch.repeat_interleave(torch.arange(4), torch.tensor(lengths)).int().cuda()

    def run(tokens, offset=0):
        flat = torch.full((n * heads * v_dim + 8,), 9.0, device="cuda", dtype=torch.bfloat16)
        out = flat[offset : offset + n * heads * v_dim].view(n, heads * v_dim)
        ops.latent_prompt(q, out, heads, key_dim, v_dim, positions, seqs, tables, pool, page, window, 0.1, tokens=tokens)
        assert bool((flat[:offset] == 9.0).all()) and bool((flat[offset + n * heads * v_dim :] == 9.0).all())
        return out

    want = run(0)
    assert bool(torch.isfinite(want.float()).all())
    for tokens in {1, max(1, most // 2), max(1, most - 1), most}:
        assert torch.equal(run(tokens), want)
    assert torch.equal(run(0, offset=1), want)
    with pytest.raises(KernelError):
        run(most + 1)


def test_tokens_and_shares_of_a_step():
    """Short portions spread over the chip, long prompts fill workgroups, shares stop at twice the compute units."""
    from types import SimpleNamespace

    import numpy as np

    from shrike_amd.engine.context import StepShape
    from shrike_amd.parts.attention import compute_units
    from shrike_amd.parts.latent_attention import LatentAttention

    part = LatentAttention.__new__(LatentAttention)
    part.spec = SimpleNamespace(num_heads=28, kv_rank=448, rot_dim=64, window=None, chunk=None)
    part.mfma, part.prompt_tokens = True, 4

    def plan(lens, starts):
        shape = StepShape(np.array(lens), np.array(starts), 16)
        part.prepare(shape)
        (note,) = shape.notes.values()
        return note

    assert compute_units() == 256
    assert plan([1501], [0]) == (1, 1, 0, 1, 4)
    assert plan([64], [0]) == (1, 1, 0, 1, 1)
    assert plan([16], [2000]) == (1, 1, 0, 16, 1)
    assert plan([2] * 60, [300] * 60)[4] == 1
    assert plan([1, 1, 300], [900, 40, 0]) == (8, 1, 2, 4, 4)
