"""bfloat16 products of more than 64 tokens with aligned rows: every tile, the ends of k, of the rows and of the
tokens, shares of k, and every way in which results leave."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from shrike_amd.kernels import ops

    return ops


def operands(n, m, k, seed=0, matrices=1):
    gen = torch.Generator("cuda").manual_seed(seed + n + 3 * m + 7 * k)
    x = torch.randn(n, k, generator=gen, device="cuda").to(BF16)
    ws = [(torch.randn(m, k, generator=gen, device="cuda") / math.sqrt(k)).to(BF16) for _ in range(matrices)]
    return x, ws


def check(out, want, k):
    """float32 sums of k products of bfloat16 numbers: an error of k 2^-24 of the sum of their magnitudes (about
    sqrt(k) of a sum's size) at the very most, and half a unit of bfloat16 where that is what is stored."""
    rel = 2.0**-8 if out.dtype == BF16 else 0.0
    bound = want.abs() * rel + want.abs().max() * (1e-6 + k * 2.0**-24)
    bad = (out.double() - want).abs() > bound
    assert not bad.any(), f"{int(bad.sum())} values off, the most by {float((out.double() - want).abs().max())}"


# (the tiles that the plan takes: weight rows x tokens)
SIZES = [
    (65, 200, 136),       # 128 x 128
    (640, 9000, 136),     # 256 x 128
    (1665, 4616, 136),    # 256 x 256
    (513, 9000, 520),     # 128 x 192
    (1665, 4616, 520),    # 192 x 192
    (1282, 7000, 520),    # 256 x 192
    (961, 9000, 1096),    # 192 x 256
    (2048, 3584, 128),    # 128 x 256
    (1281, 12000, 136),   # two products: 256 x 256, then 128 x 128
    (1281, 12000, 520),   # 192 x 192, then 256 x 128
    (1921, 9000, 1096),   # 192 x 256, then 128 x 192
    (2561, 7000, 1096),   # 256 x 192, then 128 x 128
    # k: one piece, less than a tile, a tile, a stage, a stage and a piece, three tiles, five stages and a half
    (70, 2064, 8), (70, 2064, 24), (129, 2064, 32), (129, 2064, 64), (200, 2064, 72), (300, 2064, 96), (130, 2064, 352),
    # rows that are no whole pieces, fewer than a block, one block
    (100, 3000 - 1, 64), (127, 2049, 160), (100, 80, 520), (193, 84, 1032),
]


@pytest.mark.parametrize("n, m, k", SIZES)
def test_plain_products(ops, n, m, k):
    x, (w,) = operands(n, m, k)
    wt, want = ops.retile_weight(w), x.double() @ w.double().T
    out = torch.full((n, m), float("nan"), device="cuda", dtype=BF16)
    ops.gemm_tiled_weight(x, wt, m, k, out)
    check(out, want, k)
    # a bias, float32 results in rows of a wider buffer that are no whole 16-byte pieces
    bias = torch.randn(m, generator=torch.Generator("cuda").manual_seed(m), device="cuda")
    wide = torch.full((n, m + 5), 5.0, device="cuda")
    ops.gemm_tiled_weight(x, wt, m, k, wide[:, 2 : m + 2], bias=bias)
    check(wide[:, 2 : m + 2], want + bias.double(), k)
    assert (wide[:, :2] == 5).all() and (wide[:, m + 2 :] == 5).all()
    out32 = torch.full((n, m), 2.0, device="cuda")
    ops.gemm_tiled_weight(x, wt, m, k, out32, accumulate=True)
    check(out32, want + 2.0, k)
    ops.gemm_tiled_weight(x, wt, m, k, out, bias=bias, activation="relu_squared")
    check(out, (want + bias.double()).relu().square(), 4 * k)
    ops.gemm_tiled_weight(x, wt, m, k, out, activation=("silu", m // 2 + 1))
    silu = torch.cat([torch.nn.functional.silu(want[:, : m // 2 + 1]), want[:, m // 2 + 1 :]], 1)
    check(out, silu, 2 * k)


@pytest.mark.parametrize("n, m, k", [(65, 200, 136), (640, 4500, 136), (1665, 2308, 136), (513, 4500, 520), (961, 4500, 1096),
                                     (1282, 3500, 520), (1665, 2308, 520), (500, 9475, 1024), (70, 1032, 8), (200, 1036, 96), (129, 2051, 72)])
def test_gated_products(ops, n, m, k):
    x, (g, u) = operands(n, m, k, matrices=2)
    wt = ops.interleave_gate_up(g, u)
    a, b = x.double() @ g.double().T, x.double() @ u.double().T
    out = torch.full((n, m), float("nan"), device="cuda", dtype=BF16)
    ops.gemm_tiled_weight(x, wt, m, k, out, gated=True)
    check(out, torch.nn.functional.silu(a) * b, 4 * k)
    args = torch.tensor([0.5, 1.0], device="cuda")
    ops.gemm_tiled_weight(x, wt, m, k, out, gated="quick_gelu", gate_args=args)
    a, b = a.clamp(max=0.5), b.clamp(-0.5, 0.5) + 1.0
    check(out, a * torch.sigmoid(1.702 * a) * b, 4 * k)


@pytest.mark.parametrize("n, m, k, splits", [(70, 3584, 4096, 7), (300, 200, 1048, 3), (512, 4608, 1032, 2), (513, 2060, 520, 16), (130, 2049, 96, 3)])
def test_shares_of_k(ops, n, m, k, splits):
    """Among them more shares than stages of 64: those are zeros."""
    x, (w,) = operands(n, m, k)
    parts = torch.full((splits, n, m), float("nan"), device="cuda")
    ops.gemm_tiled_weight(x, ops.retile_weight(w), m, k, parts, splits=splits)
    check(parts.sum(0), x.double() @ w.double().T, 2 * k)


def test_rows_do_not_depend_on_the_others_or_on_the_tile(ops):
    """One order of summation in every tile."""
    m, k = 9000, 1096
    x, (w,) = operands(1921, m, k)
    wt = ops.retile_weight(w)
    whole = torch.empty(1921, m, device="cuda")
    ops.gemm_tiled_weight(x, wt, m, k, whole)
    for n in (65, 192, 513, 961):
        part = torch.empty(n, m, device="cuda")
        ops.gemm_tiled_weight(x[100 : 100 + n], wt, m, k, part)
        assert torch.equal(part, whole[100 : 100 + n])
    # rows that lie further apart than k, infinities beyond them
    apart = torch.full((513, k + 24), float("inf"), device="cuda", dtype=BF16)
    apart[:, :k] = x[:513]
    part = torch.empty(513, m, device="cuda")
    ops.gemm_tiled_weight(apart[:, :k], wt, m, k, part)
    assert torch.equal(part, whole[:513])
