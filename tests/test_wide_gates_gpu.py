"""Gated products of many tokens with every gate and its constants: the same bits from registers in whole pieces as through the loop that
finishes rows of unaligned outputs, and against float64."""

import pytest
import torch

pytestmark = pytest.mark.gpu

ACTS = {"silu": lambda v: v * torch.sigmoid(v), "gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh"),
        "relu": torch.relu, "quick_gelu": lambda v: v * torch.sigmoid(1.702 * v)}


@pytest.mark.parametrize("args", [None, (0.0, 1.0), (0.7, 0.0)])
@pytest.mark.parametrize("act", ACTS)
@pytest.mark.parametrize("n, m, k", [(65, 200, 136), (513, 4504, 136), (1282, 3504, 520)])
def test_gates_in_registers(n, m, k, act, args):
    from shrike_amd.kernels import ops

    torch.manual_seed(n + m)
    x = torch.randn(n, k, device="cuda").bfloat16()
    g, u = ((torch.randn(m, k, device="cuda") / k**0.5).bfloat16() for _ in range(2))
    wt, given = ops.interleave_gate_up(g, u), None if args is None else torch.tensor(args, device="cuda")

    def run(offset):
        flat = torch.full((n * m + 8,), 5.0, device="cuda", dtype=torch.bfloat16)
        out = flat[offset : offset + n * m].view(n, m)
        ops.gemm_tiled_weight(x, wt, m, k, out, gated=act, gate_args=given)
        assert bool((flat[:offset] == 5.0).all()) and bool((flat[offset + n * m :] == 5.0).all())
        return out

    out = run(0)
    assert torch.equal(out, run(4))
    a, b = x.double() @ g.double().t(), x.double() @ u.double().t()
    if args and args[0] > 0.0:
        a, b = a.clamp(max=args[0]), b.clamp(-args[0], args[0])
    want = ACTS[act](a) * (b + (args[1] if args else 0.0))
    # float32 sums of k products and exp(), then one rounding to eight significant bits
    assert bool(((out.double() - want).abs() <= 2.0**-8 * want.abs() + 1e-5 * k**0.5).all())
