"""Experts' products in tiles of 128 or 256 weight rows x 128 or 192 pairs: lists of no pair, one, a whole tile and one
more, features that end within a tile, every form of expert, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width, ff, counts", [
    (64, 64, [0, 1, 128, 129, 385, 64]),
    (192, 320, [700, 0, 0]),
    (1344, 448, [131, 255, 257, 5, 0, 96, 512, 1]),
    (128, 192, [0] * 70 + [900, 127] + [64] * 75),  # more experts than a wavefront has lanes
    # (small matrices take the kernels for short lists up to here, see fills_long_lists)
    (64, 64, [0, 1, 128, 129, 385, 64, 36000]),
    (192, 320, [4000, 0, 0]),
    (128, 192, [0] * 70 + [900, 127] + [64] * 75 + [5000]),
])
@pytest.mark.parametrize("form", ["silu", "bounded", "single"])
def test_lists_of_every_length(width, ff, counts, form):
    from shrike_amd.kernels import ops

    torch.manual_seed(width + ff)
    experts, top = len(counts), 2
    owners = torch.repeat_interleave(torch.arange(experts), torch.tensor(counts))
    n = max(-(-owners.numel() // 1), 32 * experts)  # (an identity expert fills what is left of a token's choices)
    owners = owners[torch.randperm(owners.numel())]
    chosen = torch.full((n, top), experts, dtype=torch.int32)
    chosen[: owners.numel(), 0] = owners.int()
    dev = lambda t: t.to("cuda")  # noqa: E731
    x = dev(torch.randn(n, width).bfloat16())
    w_up, w_down = dev((torch.randn(experts, ff, width) / width**0.5).bfloat16()), dev((torch.randn(experts, width, ff) / ff**0.5).bfloat16())
    w_gate = w_up if form == "single" else dev((torch.randn(experts, ff, width) / width**0.5).bfloat16())
    weights = dev(torch.rand(n, top))
    limit, shift = (0.7, 1.0) if form == "bounded" else (None, 0.0)
    act = {"silu": "silu", "bounded": "quick_gelu", "single": "relu"}[form]
    out = torch.full((n, width), 5.0, device="cuda", dtype=torch.bfloat16)
    act_buf = torch.full((n * top, ff), float("nan"), device="cuda", dtype=torch.bfloat16)
    scratch = torch.full((ops.moe_grouped_scratch_bytes(n, width, experts, top),), 255, device="cuda", dtype=torch.uint8)
    assert n * top >= 64 * experts, "the lists are long enough for the tiles"
    up_t, down_t = ops.tile_experts(w_up), ops.tile_experts(w_down)
    gate_t = up_t if form == "single" else ops.tile_experts(w_gate)
    ops.moe_experts(x, dev(chosen), weights, gate_t, up_t, down_t, act_buf, out, act, scratch=scratch, identity=1, limit=limit,
                    up_shift=shift, tiled=True)
    want = weights.double()[:, 1, None] * x.double()
    size = want.abs()
    for e in range(experts):
        at = dev((chosen[:, 0] == e).nonzero().flatten())
        if at.numel() == 0:
            continue
        g, u = x[at].double() @ w_gate[e].double().t(), x[at].double() @ w_up[e].double().t()
        if limit:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        a = {"silu": lambda v: v * torch.sigmoid(v), "quick_gelu": lambda v: v * torch.sigmoid(1.702 * v), "relu": torch.relu}[act](g)
        h = a * (u + shift)
        w = weights.double()[at, 0, None]
        want[at] += w * (h @ w_down[e].double().t())
        size[at] += w * (h.abs() @ w_down[e].double().abs().t())
    rest = dev((chosen[:, 0] == experts).nonzero().flatten())
    want[rest] += weights.double()[rest, 0, None] * x[rest].double()
    size[rest] += (weights.double()[rest, 0, None] * x[rest].double()).abs()
    # short lists: the same sums from tiles as from rows
    few = torch.full((5, top), experts, dtype=torch.int32)  # (experts > 1: 10 pairs are few)
    few[:, 1] = torch.arange(5) % experts
    both = []
    for tiled, (g, u, d) in ((True, (gate_t, up_t, down_t)), (False, (w_gate, w_up, w_down))):
        small = torch.full((5, width), 5.0, device="cuda", dtype=torch.bfloat16)
        ops.moe_experts(x[:5], dev(few), weights[:5], g, u, d, act_buf, small, act, scratch=scratch, identity=1, limit=limit,
                        up_shift=shift, tiled=tiled)
        both.append(small)
    assert torch.equal(*both)
    # the activations are rounded to bfloat16, the result once more: eight significant bits, so 2^-8 of each at most, together
    # 2^-7 where one activation makes the result (a few in a million elements come above 2^-8); float32 sums add little
    assert bool(((out.double() - want).abs() <= 2.0**-7 * size + 1e-3).all())


@pytest.mark.parametrize("off_add, off_out", [(1, 0), (0, 1), (3, 5)])
@pytest.mark.parametrize("n, width, ff, tiled", [(6, 128, 64, True), (300, 64, 64, True), (6, 72, 40, False)])
def test_added_rows_and_results_anywhere_in_memory(n, width, ff, tiled, off_add, off_out):
    """`add` and `out` need not be 16-byte aligned: the same bits as where they are."""
    from shrike_amd.kernels import ops

    torch.manual_seed(n + width)
    experts, top = 4, 2
    x = torch.randn(n, width, device="cuda").bfloat16()
    matrices = [torch.randn(experts, r, c, device="cuda").bfloat16() for r, c in ((ff, width), (ff, width), (width, ff))]
    if tiled:
        matrices = [ops.tile_experts(w) for w in matrices]
    chosen, weights = torch.randint(0, experts + 1, (n, top), device="cuda").int(), torch.rand(n, top, device="cuda")
    added = torch.randn(n, width, device="cuda").bfloat16()
    scratch = torch.empty(ops.moe_grouped_scratch_bytes(n, width, experts, top), device="cuda", dtype=torch.uint8)
    act_buf = torch.empty(n * top, ff, device="cuda", dtype=torch.bfloat16)

    def run(off_add, off_out):
        add = torch.zeros(n * width + 16, device="cuda", dtype=torch.bfloat16)[off_add : off_add + n * width].view(n, width)
        add.copy_(added)
        flat = torch.full((n * width + 16,), 5.0, device="cuda", dtype=torch.bfloat16)
        out = flat[off_out : off_out + n * width].view(n, width)
        ops.moe_experts(x, chosen, weights, *matrices, act_buf, out, "silu", add=add, scratch=scratch, identity=1, tiled=tiled)
        assert bool((flat[:off_out] == 5.0).all()) and bool((flat[off_out + n * width :] == 5.0).all())
        return out

    assert torch.equal(run(off_add, off_out), run(0, 0))


# width, features, lists (the edges of tiles of 128 and of 192 pairs; matrices that end within a tile) and the tiles of both products
TILES = [
    (576, 192, [191, 192, 193, 384, 385, 1, 0, 7654], ("silu", "bounded"), ((256, 192), (256, 128))),
    (1344, 64, [191, 193, 0, 385, 3200], ("silu", "bounded"), ((128, 192), (256, 192))),
    (64, 704, [127, 128, 129, 191, 192, 193, 385, 2700], ("silu",), ((256, 128), (128, 192))),
    (1344, 320, [191, 192, 193, 384, 385, 1, 0, 7654], ("single",), ((256, 192), (256, 128))),
    (1344, 64, [191, 192, 193, 385, 0, 257, 63, 2719], ("single",), ((128, 192), (256, 192))),
]


@pytest.mark.parametrize("width, ff, counts, form, tiles", [(w, f, c, form, t) for w, f, c, forms, t in TILES for form in forms])
def test_every_tile(width, ff, counts, form, tiles):
    from shrike_amd.kernels import ops

    n = max(sum(counts), 32 * len(counts))
    assert ops.moe_experts_tiles(n, width, ff, len(counts), 2, 1, form == "single") == tiles
    test_lists_of_every_length(width, ff, counts, form)


def test_more_than_two_to_the_31_activations():
    """Offsets that no longer fit 32 bits: the tokens are taken in turns, by the kernel that takes fewer of them, and a token's
    result is the same bits whatever the call holds beside it."""
    from shrike_amd.kernels import ops

    width, ff, experts, top, n, few = 64, 8192, 2, 2, 131200, 20000
    assert n * top * ff > 1 << 31 and ops.moe_experts_tiles(n, width, ff, experts, top, 1) and ops.moe_experts_tiles(few, width, ff, experts, top, 1)
    gen = torch.Generator("cuda").manual_seed(1)
    x = torch.randn(n, width, generator=gen, device="cuda").bfloat16()
    w_gate, w_up = ((torch.randn(experts, ff, width, generator=gen, device="cuda") / 8).bfloat16() for _ in range(2))
    w_down = (torch.randn(experts, width, ff, generator=gen, device="cuda") / 90).bfloat16()
    tiled = [ops.tile_experts(w) for w in (w_gate, w_up, w_down)]
    chosen = torch.rand(n, experts + 1, generator=gen, device="cuda").argsort(1)[:, :top].int().contiguous()  # (no expert twice)
    weights, add = torch.rand(n, top, generator=gen, device="cuda"), torch.randn(n, width, generator=gen, device="cuda").bfloat16()
    share = torch.randn(n, 3, generator=gen, device="cuda")

    def run(lo, hi):
        rows, out = slice(lo, hi), torch.full((hi - lo, width), 5.0, device="cuda", dtype=torch.bfloat16)
        act_buf = torch.empty((hi - lo) * top, ff, device="cuda", dtype=torch.bfloat16)
        scratch = torch.empty(ops.moe_grouped_scratch_bytes(hi - lo, width, experts, top), device="cuda", dtype=torch.uint8)
        ops.moe_experts(x[rows], chosen[rows], weights[rows], *tiled, act_buf, out, "silu", scratch=scratch, add=add[rows],
                        add_gate=share[rows, 1], identity=1, tiled=True)
        return out

    out = run(0, n)
    for lo in (0, n // 2 - few // 2, n - few):
        assert torch.equal(out[lo : lo + few], run(lo, lo + few))
    for t in (0, n // 2 - 1, n // 2, n - 1):
        want = torch.sigmoid(share[t, 1].double()) * add[t].double()
        for k in range(top):
            e = int(chosen[t, k])
            y = x[t].double()
            if e < experts:
                g, u = w_gate[e].double() @ y, w_up[e].double() @ y
                y = w_down[e].double() @ (g * torch.sigmoid(g) * u)
            want += weights[t, k].double() * y
        # 2^-8 of the result and of each of 8,192 activations, whose errors add as their squares do
        assert float((out[t].double() - want).norm()) <= 2.0**-7 * float(want.norm())
