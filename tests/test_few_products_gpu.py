"""Products of few tokens that add to the stream, divide by a row's root mean square, or rotate and store what they form,
at the edges of tiles, batches and layouts, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def pieces(x):
    """[n, k] as [k / 8, n, 8]."""
    return x.view(x.shape[0], -1, 8).transpose(0, 1).contiguous()


def rows(x):
    return x.transpose(0, 1).reshape(x.shape[1], -1)


def sums_bound(k):
    """Of a float32 sum over k, to its terms' sum: one rounding a step of 32 (whose own order is the matrix unit's: 40 more)."""
    return (k / 32 + 40) * 2.0**-24


@pytest.mark.parametrize("n", [1, 3, 16, 17, 33, 64])
@pytest.mark.parametrize("m, k", [(16, 8), (48, 32), (64, 1000), (896, 896), (896, 4864), (2064, 328), (4096, 1320)])
def test_a_product_that_adds_to_the_stream(m, k, n):
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k + n)
    a = torch.randn(n, k, device="cuda").bfloat16()
    w = (torch.randn(m, k, device="cuda") / k**0.5).bfloat16()
    bias, weight = torch.randn(m, device="cuda"), 1 + 0.1 * torch.randn(m, device="cuda")
    before = torch.randn(n, m, device="cuda")
    wt, count = ops.retile_weight(w), ops.few_stream_sums(n, m, k)
    if count == 0:
        assert n > 16 and m * k > 5_000_000
        return
    for b, x in ((None, a), (bias, pieces(a)), (None, torch.cat([a, a], 1)[:, :k])):  # (the last: rows that are further apart)
        resid, out = before.clone(), torch.empty(m // 8, n, 8, device="cuda", dtype=torch.bfloat16)
        sums = torch.full((count, n), float("nan"), device="cuda")
        if x.dim() == 2 and x.stride(0) % 8:
            continue
        ops.few_stream(x, wt, m, k, resid, weight, out, sums, bias=b)
        want = before.double() + a.double() @ w.double().t() + (0 if b is None else b.double())
        size = before.double().abs() + a.double().abs() @ w.double().abs().t() + (0 if b is None else b.double().abs())
        assert bool(((resid.double() - want).abs() <= (sums_bound(k) + 2.0**-22) * size).all())
        # what the next product gets comes from the stream as it was stored: one rounding to bfloat16, one of the product before
        scaled = resid.double() * weight.double()
        assert bool(((rows(out).double() - scaled).abs() <= (2.0**-8 + 2.0**-23) * scaled.abs()).all())
        squares = (resid.double() ** 2).view(n, count, -1).sum(-1).t()
        assert bool(((sums.double() - squares).abs() <= 8 * 2.0**-24 * squares).all())


def test_matrices_that_it_does_not_take():
    from shrike_amd.kernels import ops

    assert [ops.few_stream_sums(n, m, k) for n, m, k in ((8, 5120, 5120), (8, 24, 64), (8, 896, 100), (17, 1536, 8960), (65, 16, 64))] == [0] * 5
    a, w = torch.zeros(65, 64, device="cuda").bfloat16(), torch.zeros(16, 64, device="cuda").bfloat16()
    with pytest.raises(ops.KernelError):
        ops.few_stream(a, ops.retile_weight(w), 16, 64, torch.zeros(65, 16, device="cuda"), torch.ones(16, device="cuda"),
                       torch.empty(2, 65, 8, device="cuda").bfloat16(), torch.empty(2, 65, device="cuda"))


def scaled_rows(n, k, groups):
    from shrike_amd.kernels import ops

    x, weight = 3.0 * torch.randn(n, k, device="cuda"), 1 + 0.1 * torch.randn(k, device="cuda")
    r = (x * weight).bfloat16()
    sums = (x.double() ** 2).view(n, groups, -1).sum(-1).t().contiguous().float()
    rms = torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5)
    return ops.ScaledRows(pieces(r), sums, 1e-5), r, rms


@pytest.mark.parametrize("n", [1, 16, 17, 40, 64])
@pytest.mark.parametrize("m, k, groups", [(16, 16, 1), (40, 896, 112), (37, 904, 113), (256, 1536, 192), (304, 4096, 256)])
def test_a_gated_product_of_rows_that_are_still_to_be_divided(m, k, groups, n):
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k + n)
    x, r, rms = scaled_rows(n, k, groups)
    gate, up = ((torch.randn(m, k, device="cuda") / k**0.5).bfloat16() for _ in range(2))
    wt = ops.interleave_gate_up(gate, up)
    g, u = (r.double() @ gate.double().t()) * rms, (r.double() @ up.double().t()) * rms
    gs, us = ((r.double().abs() @ t.double().abs().t()) * rms for t in (gate, up))
    want = g * torch.sigmoid(g) * u
    each = sums_bound(k) + (groups + 8) * 2.0**-24  # (the squares' sum, the root and the product with it)
    bound = 2.0**-8 * want.abs() + 2 * each * (1.1 * gs * u.abs() + us * (g * torch.sigmoid(g)).abs()) + 1e-7
    out = torch.full((n, m + 8), 7.0, device="cuda", dtype=torch.bfloat16)
    ops.few_gated(x, wt, m, k, out[:, :m], "silu")
    assert bool(((out[:, :m].double() - want).abs() <= bound).all()) and bool((out[:, m:] == 7.0).all())
    if m % 8 == 0:
        inside = torch.empty(m // 8, n, 8, device="cuda", dtype=torch.bfloat16)
        ops.few_gated(x, wt, m, k, inside, "silu")
        assert torch.equal(rows(inside), out[:, :m])


@pytest.mark.parametrize("n", [1, 7, 16, 17, 50, 65, 400, 512])
@pytest.mark.parametrize("heads, kv_heads, head_dim, k", [(14, 2, 64, 896), (3, 1, 16, 8), (4, 4, 128, 1000), (2, 1, 48, 3584)])
@pytest.mark.parametrize("scaled, write_kv", [(True, True), (False, True), (True, False)])
def test_projections_that_are_rotated_and_stored(heads, kv_heads, head_dim, k, n, scaled, write_kv):
    from shrike_amd.kernels import ops

    torch.manual_seed(heads + k + n)
    dev, page_size = torch.device("cuda"), 16
    width, half = (heads + 2 * kv_heads) * head_dim, head_dim // 2
    x, r, rms = scaled_rows(n, k, k // (8 if k <= 2048 else 16))
    if not scaled:
        x, rms = r, torch.ones(n, 1, device=dev, dtype=torch.float64)
    w, bias = (torch.randn(width, k, device=dev) / k**0.5).bfloat16(), torch.randn(width, device=dev)
    positions = torch.tensor([(37 * i) % 50 for i in range(n)], dtype=torch.int32, device=dev)
    token_seq = torch.arange(n - 1, -1, -1, dtype=torch.int32, device=dev)
    tables = torch.randperm(4 * n, device=dev).to(torch.int32).view(n, 4)
    inv_freq = 1.0 / (1e4 ** (torch.arange(0, head_dim, 2, device=dev).float() / head_dim))
    pool = ops.key_pool_shape(4 * n, kv_heads, page_size, head_dim)
    k_pool = torch.full(pool, 3.0, device=dev, dtype=torch.bfloat16)
    v_pool = torch.full((4 * n, kv_heads, head_dim, page_size), 3.0, device=dev, dtype=torch.bfloat16)
    out = torch.full((n, width), 5.0, device=dev, dtype=torch.bfloat16)
    ops.few_heads(x, ops.retile_weight(w), k, out, heads, kv_heads, head_dim, inv_freq, positions, token_seq, tables, k_pool,
                  v_pool, page_size, write_kv=write_kv, bias=bias, magnitude=1.25)

    p = ((r.double() @ w.double().t()) * rms + bias.double()).view(n, heads + 2 * kv_heads, head_dim)
    size = ((r.double().abs() @ w.double().abs().t()) * rms + bias.double().abs()).view_as(p)
    angle = (positions.float()[:, None] * inv_freq).double()[:, None]
    lo, hi = p[..., :half], p[..., half:]
    turned = 1.25 * torch.cat([lo * angle.cos() - hi * angle.sin(), hi * angle.cos() + lo * angle.sin()], -1)
    # both partners' sums, and 2^-22 for sine and cosine; half an ulp of bfloat16
    both = (sums_bound(k) + (k // 8 + 12) * 2.0**-24) * 1.25 * (size + torch.cat([size[..., half:], size[..., :half]], -1))

    def close(got, want, allowed):
        return bool(((got.double() - want).abs() <= 2.0**-8 * want.abs() + allowed + 1e-7).all())

    assert close(out.view_as(p)[:, :heads], turned[:, :heads], both[:, :heads])
    assert bool((out.view_as(p)[:, heads:] == 5.0).all())
    page = tables[token_seq.long(), (positions // page_size).long()].long()
    slot = (positions % page_size).long()
    slab = ops.key_slab(head_dim)
    keys = k_pool.permute(0, 3, 1, 2, 4).reshape(4 * n, page_size, kv_heads, head_dim)
    values = v_pool.permute(0, 3, 1, 2)
    assert k_pool.shape[-1] == slab
    stored = torch.zeros(4 * n, page_size, dtype=torch.bool, device=dev)
    if write_kv:
        stored[page, slot] = True
        assert close(keys[page, slot], turned[:, heads : heads + kv_heads], both[:, heads : heads + kv_heads])
        assert close(values[page, slot], p[:, heads + kv_heads :], both[:, heads + kv_heads :])
    assert bool((keys[~stored] == 3.0).all()) and bool((values[~stored] == 3.0).all())


def test_a_token_does_not_see_the_others():
    """Bit for bit: also beside rows of infinities."""
    from shrike_amd.kernels import ops

    torch.manual_seed(0)
    m, k = 896, 1000
    a = torch.randn(16, k, device="cuda").bfloat16()
    wt, weight = ops.retile_weight((torch.randn(m, k, device="cuda") / 30).bfloat16()), torch.ones(m, device="cuda")

    def run(x):
        n = x.shape[0]
        resid, out = torch.zeros(n, m, device="cuda"), torch.empty(m // 8, n, 8, device="cuda", dtype=torch.bfloat16)
        sums = torch.empty(ops.few_stream_sums(n, m, k), n, device="cuda")
        ops.few_stream(x, wt, m, k, resid, weight, out, sums)
        return resid, rows(out), sums.t()

    whole, few = run(a), run(a[3:9])
    wild = a.clone()
    wild[0], wild[15] = float("inf"), float("nan")
    for one, six, beside in zip(whole, few, run(wild)):
        assert torch.equal(one[1:15], beside[1:15])
        assert torch.equal(one[3:9], six)
