"""The gated product of few tokens with every gate: activations, and limits and a shift that apply to what has been divided by the root mean
square, against float64."""

import pytest
import torch

from .test_few_products_gpu import pieces, sums_bound

pytestmark = pytest.mark.gpu

ACTIVATIONS = {"silu": lambda z: z * torch.sigmoid(z), "quick_gelu": lambda z: z * torch.sigmoid(1.702 * z), "relu": torch.relu,
               "gelu_tanh": lambda z: torch.nn.functional.gelu(z, approximate="tanh")}


@pytest.mark.parametrize("n", [1, 16, 40])
@pytest.mark.parametrize("activation", sorted(ACTIVATIONS))
@pytest.mark.parametrize("limit, shift", [(None, 0.0), (1.0, 0.0), (0.6, 1.0), (None, -0.5)])
@pytest.mark.parametrize("size", [5.0, 0.1])  # undivided, most products are beyond the limit, or none is
def test_the_gate_of_divided_products(n, activation, limit, shift, size):
    from shrike_amd.kernels import ops

    m, k, groups = 72, 904, 113
    torch.manual_seed(n + len(activation))
    x, weight = size * torch.randn(n, k, device="cuda"), 1 + 0.1 * torch.randn(k, device="cuda")
    r = (x * weight).bfloat16()
    sums = (x.double() ** 2).view(n, groups, -1).sum(-1).t().contiguous().float()
    rms = torch.rsqrt((x.double() ** 2).mean(1, keepdim=True) + 1e-5)
    gate, up = ((torch.randn(m, k, device="cuda") / k**0.5).bfloat16() for _ in range(2))
    args = None if limit is None and shift == 0.0 else torch.tensor([limit or 0.0, shift], device="cuda")
    out = torch.empty(n, m, device="cuda", dtype=torch.bfloat16)
    ops.few_gated(ops.ScaledRows(pieces(r), sums, 1e-5), ops.interleave_gate_up(gate, up), m, k, out, activation, args)

    g, u = (r.double() @ gate.double().t()) * rms, (r.double() @ up.double().t()) * rms
    gs, us = ((r.double().abs() @ t.double().abs().t()) * rms for t in (gate, up))
    if limit is not None:
        assert bool((u.abs() > limit).any()) and bool((u.abs() < limit).any())
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    a = ACTIVATIONS[activation](g)
    want = a * (u + shift)
    # both sums, the squares', the root and the product with it; slopes of at most 1.2; the exponential's 2^-20 and one rounding to bfloat16
    each = sums_bound(k) + (groups + 8) * 2.0**-24
    bound = (2.0**-8 + 2.0**-20) * want.abs() + 2 * each * (1.2 * gs * (u + shift).abs() + us * a.abs()) + 1e-6
    assert bool(((out.double() - want).abs() <= bound).all())
