"""Products with matrices of few rows over many tokens, and batched products in each of their shapes, against
float64, at the edges of tiles and with ends of k that are no whole step."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65, 80, 1501])
@pytest.mark.parametrize("m, k", [(1, 64), (10, 3584), (16, 896), (17, 72), (64, 520), (65, 512)])
def test_few_rows_many_tokens(n, m, k):
    from shrike_amd.kernels import ops

    torch.manual_seed(n + m + k)
    a, w = torch.randn(n, k, device="cuda").bfloat16(), torch.randn(m, k, device="cuda").bfloat16()
    bias, wt = torch.randn(m, device="cuda"), ops.retile_weight(w)
    want = a.double() @ w.double().t() + bias.double()
    out = torch.full((n, m + 3), 7.0, device="cuda")
    ops.gemm_tiled_weight(a, wt, m, k, out[:, :m], bias=bias)
    # float32 sums: at most k / 32 + 40 roundings of half an ulp of a partial sum each
    size = a.double().abs() @ w.double().abs().t() + bias.double().abs()
    assert bool(((out[:, :m].double() - want).abs() <= (k / 32 + 40) * 2.0**-24 * size).all())
    assert bool((out[:, m:] == 7.0).all())
    half = torch.empty(n, m, device="cuda", dtype=torch.bfloat16)
    ops.gemm_tiled_weight(a, wt, m, k, half, bias=bias)
    assert torch.equal(half, out[:, :m].bfloat16())
    few = torch.empty(n - 3, m, device="cuda", dtype=torch.bfloat16)
    if n - 3 > 64:
        ops.gemm_tiled_weight(a[3:], wt, m, k, few, bias=bias)
        assert torch.equal(few, half[3:])


@pytest.mark.parametrize("m, k", [(896, 896), (1152, 896), (256, 40), (896, 4864), (1000, 2056), (300, 8192)])
def test_small_matrices_without_staging(m, k):
    """Every tile that serves small matrices from 17 tokens on (and what serves them beyond), whole and in shares."""
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k)
    n_max = 1200
    a, w = torch.randn(n_max, k, device="cuda").bfloat16(), torch.randn(m, k, device="cuda").bfloat16()
    bias, wt = torch.randn(m, device="cuda"), ops.retile_weight(w)
    want = a.double() @ w.double().t()
    size = a.double().abs() @ w.double().abs().t()
    bound = (k / 32 + 48) * 2.0**-24
    for n in (17, 32, 33, 64, 65, 128, 129, 256, 300, 511, 1200):
        out = torch.full((n, m), 7.0, device="cuda")
        ops.gemm_tiled_weight(a[:n], wt, m, k, out, bias=bias)
        off = (out.double() - want[:n] - bias.double()).abs()
        assert bool((off <= bound * (size[:n] + bias.double().abs())).all()), n
        half = torch.empty(n, m, device="cuda", dtype=torch.bfloat16)
        ops.gemm_tiled_weight(a[:n], wt, m, k, half, bias=bias)
        assert torch.equal(half, out.bfloat16()), n
        splits = max(2, ops.gemm_splits(n, m, k))
        parts = torch.full((splits, n, m), float("nan"), device="cuda")
        ops.gemm_tiled_weight(a[:n], wt, m, k, parts, splits=splits)
        assert bool(((parts.double().sum(0) - want[:n]).abs() <= bound * size[:n]).all()), n
        if n == 64:  # a captured step stands for every batch up to its own size
            few = torch.empty(41, m, device="cuda")
            ops.gemm_tiled_weight(a[:41], wt, m, k, few, bias=bias)
            assert torch.equal(few, out[:41])


@pytest.mark.parametrize("batch, m, k", [(3, 40, 8), (28, 448, 128), (5, 130, 200), (14, 512, 256), (2, 3, 40), (1, 64, 24)])
def test_batched_products_of_every_shape(batch, m, k):
    from shrike_amd.kernels import ops

    torch.manual_seed(batch + m + k)
    n_max = 300
    a = torch.randn(n_max, batch * k + 8, device="cuda").bfloat16()
    w = torch.randn(batch, m, k, device="cuda").bfloat16()
    per = a[:, : batch * k].view(n_max, batch, k).transpose(0, 1).double()
    want = (per @ w.transpose(1, 2).contiguous().double()).transpose(0, 1).reshape(n_max, batch * m)
    size = (per.abs() @ w.transpose(1, 2).contiguous().double().abs()).transpose(0, 1).reshape(n_max, batch * m)
    whole = None
    for n in (n_max, 1, 15, 16, 17, 65, 129):
        out = torch.full((n, batch * m + 4), 7.0, device="cuda")
        ops.gemm_batched(a[:n, : batch * k], w, out[:, : batch * m], batch, k, m)
        assert bool(((out[:, : batch * m].double() - want[:n]).abs() <= (k / 32 + 40) * 2.0**-24 * size[:n]).all())
        assert bool((out[:, batch * m :] == 7.0).all())
        whole = out if whole is None else whole
        assert torch.equal(out, whole[:n]), "the same bits in every shape"
        odd = torch.full((n, batch * m + 3), 7.0, device="cuda", dtype=torch.bfloat16)  # rows no multiple of 4 elements apart
        ops.gemm_batched(a[:n, : batch * k], w, odd[:, 1 : 1 + batch * m], batch, k, m)
        assert torch.equal(odd[:, 1 : 1 + batch * m], out[:, : batch * m].bfloat16())


@pytest.mark.parametrize("m, k", [(4080, 896), (4096, 24), (4100, 896), (4864, 1024), (4864, 1032), (8176, 264)])
def test_gated_products_of_a_short_k(m, k):
    """Where 16 wavefronts share k and where four do: up to 16 tokens beside what serves each token alone."""
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k)
    a = torch.randn(16, k, device="cuda").bfloat16()
    gate, up = ((torch.randn(m, k, device="cuda") / k**0.5).bfloat16() for _ in range(2))
    wt = ops.interleave_gate_up(gate, up)
    g, u = a.double() @ gate.double().t(), a.double() @ up.double().t()
    sized = [a.double().abs() @ w.double().abs().t() for w in (gate, up)]
    act = g * torch.sigmoid(g)
    # float32 sums as above, SiLU's slope is at most 1.1; bfloat16 results (half an ulp is 2^-9, the rest for the exponential)
    each = (k / 32 + 40) * 2.0**-24
    bound = 2.0**-8 * (act * u).abs() + 2 * each * (1.1 * sized[0] * u.abs() + sized[1] * act.abs())
    whole = torch.empty(16, m, device="cuda", dtype=torch.bfloat16)
    ops.gemm_tiled_weight(a, wt, m, k, whole, gated=True)
    assert bool(((whole.double() - act * u).abs() <= bound + 1e-7).all())
    for n in (1, 5):
        out = torch.full((n, m + 8), 7.0, device="cuda", dtype=torch.bfloat16)
        ops.gemm_tiled_weight(a[16 - n:], wt, m, k, out[:, :m], gated=True)
        assert torch.equal(out[:, :m], whole[16 - n:]) and bool((out[:, m:] == 7.0).all())


@pytest.mark.parametrize("m, k, n", [(896, 896, 17), (896, 896, 64), (1152, 896, 40), (896, 4864, 65), (896, 4864, 256), (512, 3584, 300),
                                     (64, 3584, 200), (896, 4864, 33)])
def test_a_reader_of_shares_gets_small_products_unrounded(m, k, n):
    """The residual after the reading norm is off by float32 roundings only, whether k was shared or not."""
    from shrike_amd.engine.context import Workspace
    from shrike_amd.engine.runtime import Runtime
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k + n)
    runtime, space = Runtime("cuda:0", torch.bfloat16), Workspace("cuda:0")

    class Context:
        buffer = staticmethod(space.get)

    a, w = torch.randn(n, k, device="cuda").bfloat16(), torch.randn(m, k, device="cuda").bfloat16()
    bias = torch.randn(m, device="cuda")
    exact, size = a.double() @ w.double().t(), a.double().abs() @ w.double().abs().t()
    bound = (k / 32 + 48) * 2.0**-24  # (as above, and one more for the residual's own sum)
    resid = torch.randn(n, m, device="cuda")
    want = resid.double() + exact
    product = runtime.linear_deferred(Context, "p", a, runtime.weight(w))
    ops.add_rmsnorm(resid, product, torch.ones(m, device="cuda"), 1e-6, torch.empty(n, m, device="cuda").bfloat16())
    assert bool(((resid.double() - want).abs() <= bound * size + 2.0**-24 * want.abs()).all())
    product = runtime.linear_deferred(Context, "q", a, runtime.weight(w), bias=bias, reader="position")
    got = product.parts.double().sum(0) + (0 if product.bias is None else product.bias.double())
    assert bool(((got - exact - bias.double()).abs() <= bound * (size + bias.double().abs())).all())


@pytest.mark.parametrize("m, k", [(300, 64), (1152, 896), (896, 4864), (2000, 264), (37, 72)])
@pytest.mark.parametrize("n", [17, 64, 100, 200, 300, 700, 1200])
def test_small_matrices_add_to_their_output_and_activate(m, k, n):
    """Sums onto what is there, the square of ReLU and SiLU of the first columns, with a bias, in the kernels that stage nothing."""
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k + n)
    a, w = torch.randn(n, k, device="cuda").bfloat16(), (torch.randn(m, k, device="cuda") / k**0.5).bfloat16()
    bias, wt = torch.randn(m, device="cuda"), ops.retile_weight(w)
    v = a.double() @ w.double().t() + bias.double()
    off = (k / 32 + 48) * 2.0**-24 * (a.double().abs() @ w.double().abs().t() + bias.double().abs())  # of a float32 sum
    there = torch.randn(n, m + 8, device="cuda")
    for dtype, ulp in ((torch.float32, 2.0**-23), (torch.bfloat16, 2.0**-8)):
        out = there.to(dtype, copy=True)
        if dtype == torch.float32:
            ops.gemm_tiled_weight(a, wt, m, k, out[:, :m], bias=bias, accumulate=True)
            want = there[:, :m].double() + v
            assert bool(((out[:, :m].double() - want).abs() <= off + ulp * (want.abs() + off)).all())
        ops.gemm_tiled_weight(a, wt, m, k, out[:, :m], bias=bias, activation="relu_squared")
        want = v.clamp(min=0) ** 2
        assert bool(((out[:, :m].double() - want).abs() <= 2.2 * off * (v.abs() + off) + ulp * want).all())
        for rows in (1, 37, m - 3, m):
            ops.gemm_tiled_weight(a, wt, m, k, out[:, :m], bias=bias, activation=("silu", min(rows, m)))
            want = v.clone()
            want[:, :rows] = v[:, :rows] * torch.sigmoid(v[:, :rows])
            # (the slope of SiLU is at most 1.1; its float32 exponential and quotient: a few roundings of the result, or of
            # an exponent of up to 40, 2^-18)
            assert bool(((out[:, :m].double() - want).abs() <= 1.1 * off + (ulp + 2.0**-18) * want.abs() + 1e-12).all()), rows
        assert torch.equal(out[:, m:], there[:, m:].to(dtype))


@pytest.mark.parametrize("m, k", [(896, 896), (1152, 896), (896, 4864), (1000, 2056), (512, 3584), (2048, 1024), (10, 3584), (64, 520), (32, 8192)])
def test_small_products_keep_their_bits_within_a_batch_bucket(m, k):
    """A captured step of 32, 64, 128 or 256 rows stands for every smaller batch down to the next."""
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k)
    a, w = torch.randn(256, k, device="cuda").bfloat16(), torch.randn(m, k, device="cuda").bfloat16()
    wt = ops.retile_weight(w)
    for end, fewer in ((32, (17, 21)), (64, (33, 41)), (128, (65, 97)), (256, (129, 201))):
        splits = ops.gemm_splits(end, m, k)
        whole = torch.full((splits, end, m), float("nan"), device="cuda")
        ops.gemm_tiled_weight(a[:end], wt, m, k, whole if splits > 1 else whole[0], splits=splits)
        assert not bool(torch.isnan(whole).any())
        for n in fewer:
            part = torch.full((splits, n, m), float("nan"), device="cuda")
            ops.gemm_tiled_weight(a[:n], wt, m, k, part if splits > 1 else part[0], splits=splits)
            assert torch.equal(part, whole[:, :n]), (n, end)
