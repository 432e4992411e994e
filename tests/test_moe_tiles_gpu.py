"""Experts' products in tiles of 256 weight rows x 128 pairs: lists of no pair, one, a whole tile and one
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
