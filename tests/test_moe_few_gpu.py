"""The experts of up to 16 tokens with the shared one in the same launches, against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def gate(g, u, activation, limit, shift):
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    act = {"silu": lambda z: z * torch.sigmoid(z), "quick_gelu": lambda z: z * torch.sigmoid(1.702 * z),
           "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh"), "relu": torch.relu}[activation]
    return act(g) * (u + shift)


@pytest.mark.parametrize("n", [1, 2, 8, 15, 16])
@pytest.mark.parametrize("width, ff, experts, identity, top, shared, activation, limit, shift, shared_gate", [
    (64, 64, 3, 0, 1, None, "silu", None, 0.0, False),
    (64, 128, 4, 2, 2, 96, "quick_gelu", 7.0, 1.0, False),
    (320, 64, 8, 0, 8, 32, "gelu_tanh", None, 0.0, True),
    (3584, 1216, 8, 2, 2, 2432, "quick_gelu", 7.0, 1.0, False),
    (896, 1216, 60, 4, 5, 2432, "silu", None, 0.0, True),
])
def test_against_float64(n, width, ff, experts, identity, top, shared, activation, limit, shift, shared_gate):
    from shrike_amd.kernels import ops

    assert ops.moe_few_takes(n, top) and not ops.moe_few_takes(17, top) and not ops.moe_few_takes(n, 9)
    torch.manual_seed(n + width + ff)

    def matrix(*shape):
        return (torch.randn(*shape, device="cuda") / shape[-1] ** 0.5).bfloat16()

    x = torch.randn(n, width, device="cuda").bfloat16()
    gates, ups, downs = ([matrix(m, k) for _ in range(experts)] for m, k in ((ff, width), (ff, width), (width, ff)))
    chosen = torch.stack([torch.randperm(experts + identity, device="cuda")[:top] for _ in range(n)]).to(torch.int32)
    if n > 2:
        chosen[1] = chosen[0]  # (lists of more than one token)
    weights = torch.rand(n, top, device="cuda")
    more = None
    column = torch.randn(n, 3, device="cuda")
    if shared:
        sg, su, sd = matrix(shared, width), matrix(shared, width), matrix(width, shared)
        more = (ops.interleave_gate_up(sg, su), ops.retile_weight(sd), shared)
    act = torch.empty(n * top, ff, device="cuda", dtype=torch.bfloat16)
    shared_act = torch.empty(n, shared or 1, device="cuda", dtype=torch.bfloat16)
    pair_out = torch.full((n * (top + 1), width), float("nan"), device="cuda")
    out = torch.empty(n, width, device="cuda", dtype=torch.bfloat16)
    ops.moe_few(x, chosen, weights, *(ops.tile_experts(t) for t in (gates, ups, downs)), act, pair_out, out, activation, shared=more,
                shared_act=shared_act, add_gate=column[:, 1] if shared_gate else None, identity=identity, limit=limit, up_shift=shift,
                shared_limit=limit)

    want, allowed = torch.zeros(n, width, device="cuda", dtype=torch.float64), torch.zeros(n, width, device="cuda", dtype=torch.float64)
    each = (max(width, ff, shared or 0) / 32 + 40) * 2.0**-24

    def expert(rows, g, u, d, share, at):
        a = gate(rows @ g.double().t(), rows @ u.double().t(), activation, limit, shift)
        # float32 sums of the two products (a slope of at most 1.2 and the other factor), one rounding to bfloat16
        gs, us = rows.abs() @ g.double().abs().t(), rows.abs() @ u.double().abs().t()
        off = 2.0**-8 * a.abs() + 2 * each * (1.2 * gs * (us + shift) + us * gs) + 1e-9
        want[at] += share * (a @ d.double().t())
        allowed[at] += share.abs() * ((off + 2 * each * a.abs()) @ d.double().abs().t())

    xd = x.double()
    for t in range(n):
        for k in range(top):
            e, w, at = int(chosen[t, k]), weights[t, k].double(), slice(t, t + 1)
            if e >= experts:
                want[at] += w * xd[at]
            else:
                expert(xd[at], gates[e], ups[e], downs[e], w, at)
    if shared:
        share = torch.sigmoid(column[:, 1:2].double()) if shared_gate else torch.ones(n, 1, device="cuda", dtype=torch.float64)
        expert(xd, sg, su, sd, share, slice(0, n))
    assert bool(((out.double() - want).abs() <= 2.0**-8 * want.abs() + allowed + 1e-7).all())
