"""bfloat16 products of more than 64 tokens: every tile, the ends of k, of the rows and of the tokens, shares of k, and
every way in which results leave; rows that are not aligned, which a kernel of their own takes."""

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


# (the tiles that the plan takes, weight rows x tokens: TILES below)
SIZES = [
    (65, 200, 136),
    (640, 9000, 136),
    (1665, 4616, 136),
    (513, 9000, 520),
    (1665, 4616, 520),
    (1282, 7000, 520),
    (961, 9000, 1096),
    (2048, 3584, 128),
    (1281, 12000, 136),   # (two products each)
    (1281, 12000, 520),
    (1921, 9000, 1096),
    (2561, 7000, 1096),
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


# every tile as a plan takes it: (n, m, k, gated, shares): tiles of the one or two launches
TILES = {
    (65, 200, 136, False, 1): ((128, 128),),
    (640, 9000, 136, False, 1): ((256, 128),),
    (1665, 4616, 136, False, 1): ((256, 256),),
    (513, 9000, 520, False, 1): ((128, 192),),
    (1665, 4616, 520, False, 1): ((192, 192),),
    (1282, 7000, 520, False, 1): ((256, 192),),
    (961, 9000, 1096, False, 1): ((192, 256),),
    (2048, 3584, 128, False, 1): ((256, 128),),
    (1281, 12000, 136, False, 1): ((256, 256), (128, 128)),
    (1281, 12000, 520, False, 1): ((192, 192), (256, 128)),
    (1921, 9000, 1096, False, 1): ((192, 256), (128, 192)),
    (2561, 7000, 1096, False, 1): ((256, 192), (256, 128)),
    (65, 200, 136, True, 1): ((128, 128),),
    (640, 4500, 136, True, 1): ((256, 128),),
    (1665, 2308, 136, True, 1): ((256, 256),),
    (513, 4500, 520, True, 1): ((128, 192),),
    (961, 4500, 1096, True, 1): ((192, 256),),
    (1282, 3500, 520, True, 1): ((256, 192),),
    (1665, 2308, 520, True, 1): ((192, 192),),
    (512, 4608, 1032, False, 2): ((128, 192),),
    (513, 2060, 520, False, 16): ((256, 256),),
    # 128 x 256: rows that are and are no whole pieces, half a last stage of k; alone, as the second of two, with shares
    (1181, 4616, 2056, False, 1): ((128, 256),),
    (1181, 4615, 2056, False, 1): ((128, 256),),
    (2049, 9003, 2056, False, 1): ((256, 192), (128, 256)),
    (158, 9008, 2056, True, 1): ((128, 256),),
    (158, 9003, 2056, True, 1): ((128, 256),),
    (1925, 4616, 2056, True, 1): ((256, 192), (128, 256)),
    (158, 9003, 3592, False, 2): ((128, 256),),
    (1181, 2060, 2056, False, 3): ((128, 256),),
    # the others in shares of k
    (778, 4616, 72, False, 2): ((256, 256),),
    (158, 9003, 72, False, 2): ((256, 128),),
    (778, 5125, 1048, False, 2): ((256, 192),),
    (406, 9003, 2056, False, 2): ((192, 256),),
    (1026, 3589, 520, False, 2): ((192, 192),),
    (778, 2309, 1048, False, 2): ((128, 192),),
    # the tiles left that a second product may have
    (1801, 7001, 2056, True, 1): ((256, 256), (256, 192)),
    (1026, 9003, 2056, True, 1): ((256, 192), (192, 192)),
}


@pytest.mark.parametrize("n, m, k, gated, splits", TILES)
def test_every_tile(ops, n, m, k, gated, splits):
    assert ops.gemm_tiles(n, m, k, gated, splits) == TILES[n, m, k, gated, splits]
    if gated:
        test_gated_products(ops, n, m, k)
    elif splits > 1:
        test_shares_of_k(ops, n, m, k, splits)
    elif (n, m, k) not in SIZES:
        test_plain_products(ops, n, m, k)


# rows that begin anywhere: (n, m, k, gated), elements between rows beyond k; every tile of their kernel, also with more
# workgroups of 128 x 128 than compute units (four wavefronts instead of eight)
UNALIGNED = {
    (65, 130, 36, False, 0): ((128, 128),),
    (129, 516, 333, False, 0): ((128, 128),),
    (300, 1000, 520, False, 3): ((128, 128),),
    (769, 4616, 36, True, 0): ((128, 128),),
    (257, 12003, 36, False, 0): ((256, 128),),
    (129, 9003, 100, True, 4): ((256, 128),),
    (2199, 1100, 12, False, 0): ((128, 128),),  # (486 of 128 x 128 in its three shares)
    (641, 12003, 37, False, 0): ((256, 256),),
    (257, 12003, 72, True, 1): ((256, 256),),
    (1281, 12003, 1100, False, 0): ((256, 256), (128, 128)),
    (641, 12003, 1100, True, 0): ((256, 256), (128, 128)),
    (2049, 9003, 2052, True, 0): ((256, 256), (256, 128)),
}


@pytest.mark.parametrize("n, m, k, gated, apart", UNALIGNED)
def test_rows_that_are_not_aligned(ops, n, m, k, gated, apart):
    assert ops.gemm_tiles(n, m, k, gated, 1, aligned=False) == UNALIGNED[n, m, k, gated, apart]
    x, ws = operands(n, m, k, matrices=2 if gated else 1)
    rows = torch.full((n, k + apart), float("nan"), device="cuda", dtype=BF16)  # (NaN between the rows)
    rows[:, :k] = x
    rows = rows[:, :k]
    assert not ops.rows_aligned(rows) or k % 8
    first, *second = (x.double() @ w.double().T for w in ws)
    out, bias = torch.full((n, m), float("nan"), device="cuda", dtype=BF16), torch.randn(m, device="cuda")
    if gated:
        wt = ops.interleave_gate_up(*ws)
        ops.gemm_tiled_weight(rows, wt, m, k, out, gated=True)
        check(out, torch.nn.functional.silu(first) * second[0], 4 * k)
        args = torch.tensor([0.5, 1.0], device="cuda")
        ops.gemm_tiled_weight(rows, wt, m, k, out, gated="quick_gelu", gate_args=args)
        g, u = first.clamp(max=0.5), second[0].clamp(-0.5, 0.5) + 1.0
        check(out, g * torch.sigmoid(1.702 * g) * u, 4 * k)
        return
    wt = ops.retile_weight(ws[0])
    ops.gemm_tiled_weight(rows, wt, m, k, out, bias=bias)
    check(out, first + bias.double(), k)
    edge = m - 7  # (in the second of two products)
    ops.gemm_tiled_weight(rows, wt, m, k, out, activation=("silu", edge))
    check(out, torch.cat([torch.nn.functional.silu(first[:, :edge]), first[:, edge:]], 1), 2 * k)
    parts = torch.full((3, n, m), float("nan"), device="cuda")
    ops.gemm_tiled_weight(rows, wt, m, k, parts, splits=3)
    check(parts.sum(0), first, 2 * k)


@pytest.mark.parametrize("m", [2312, 2308, 2311])  # whole pieces, half a piece left, rows that begin anywhere
@pytest.mark.parametrize("n, k", [(70, 136), (513, 520)])
def test_results_are_the_same_bits_however_they_leave(ops, n, m, k):
    """In pieces straight from registers, in pieces behind the loop that finishes them, as single values."""
    x, (g, u) = operands(n, m, k, matrices=2)
    pair, plain = ops.interleave_gate_up(g, u), ops.retile_weight(g)
    wide, odd = (torch.full((n, m + extra), 3.0, device="cuda", dtype=BF16) for extra in (-m % 8 + 8, 8 + (m + 1) % 2))
    bias = torch.randn(m + 1, device="cuda")
    a, b = x.double() @ g.double().T, x.double() @ u.double().T
    gates = {"silu": lambda v: v * torch.sigmoid(v), "gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh"),
             "relu": torch.relu, "quick_gelu": lambda v: v * torch.sigmoid(1.702 * v)}

    def same(want, bound, **how):
        outs = []
        for rows in (torch.empty(n, m, device="cuda", dtype=BF16), wide[:, :m], odd[:, 4 : m + 4]):
            rows.fill_(float("nan"))
            ops.gemm_tiled_weight(x, pair if "gated" in how else plain, m, k, rows, **how)
            outs.append(rows)
        check(outs[0], want, bound)
        assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
        assert (wide[:, m:] == 3).all() and (odd[:, :4] == 3).all() and (odd[:, m + 4 :] == 3).all()

    for name, act in gates.items():
        same(act(a) * b, 4 * k, gated=name)
        limit = torch.tensor([0.25, 0.0], device="cuda")
        same(act(a.clamp(max=0.25)) * b.clamp(-0.25, 0.25), 4 * k, gated=name, gate_args=limit)
        same(act(a) * (b + 1.5), 4 * k, gated=name, gate_args=torch.tensor([0.0, 1.5], device="cuda"))
    for shift in (0, 1):  # (a bias that is and is not 16-byte aligned)
        add = bias[shift : shift + m]
        same(a + add.double(), k, bias=add)
        same((a + add.double()).relu().square(), 4 * k, bias=add, activation="relu_squared")
    same(torch.cat([gates["silu"](a[:, :1003]), a[:, 1003:]], 1), 2 * k, activation=("silu", 1003))
    sums = []
    for rows in (torch.empty(n, m, device="cuda"), torch.empty(n, m + 6 + (m + 1) % 2, device="cuda")[:, 2 : m + 2]):
        rows.fill_(2.0)
        ops.gemm_tiled_weight(x, plain, m, k, rows, accumulate=True)
        ops.gemm_tiled_weight(x, plain, m, k, rows, bias=bias[:m], accumulate=True)
        sums.append(rows)
    check(sums[0], 2 * a + 2.0 + bias[:m].double(), 2 * k)
    assert torch.equal(*sums)
