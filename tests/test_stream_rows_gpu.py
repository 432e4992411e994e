"""Products of 17 to 64 tokens: results that leave through LDS in whole rows are the same bits as those that leave one by one (outputs
that are not 16-byte aligned), and what float64 gives."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [17, 32, 33, 64])
@pytest.mark.parametrize("m, k, form", [
    (200, 136, "float32"), (1036, 520, "float32"), (20004, 72, "float32"), (40000, 64, "float32"), (66004, 40, "float32"), (65544, 72, "bfloat16"),
    (200, 136, "bfloat16"), (1032, 520, "bfloat16"), (66008, 40, "bfloat16"), (200, 136, "gated"), (20008, 72, "gated"), (40008, 72, "gated"),
    (200, 1096, "bias"), (1036, 520, "bias"), (516, 2056, "shares"), (2052, 4104, "shares"), (300, 136, "added"),
])
def test_rows_leave_whole(n, m, k, form):
    from shrike_amd.kernels import ops

    torch.manual_seed(n + m)
    x = torch.randn(n, k, device="cuda").bfloat16()
    g, u = ((torch.randn(m, k, device="cuda") / k**0.5).bfloat16() for _ in range(2))
    bias = torch.randn(m, device="cuda") if form == "bias" else None
    wt = ops.interleave_gate_up(g, u) if form == "gated" else ops.retile_weight(g)
    shape = (5, n, m) if form == "shares" else (n, m)
    dtype = torch.bfloat16 if form in ("bfloat16", "gated") else torch.float32
    size = n * m * (5 if form == "shares" else 1)

    def run(offset):
        flat = torch.full((size + 8,), 5.0, device="cuda", dtype=dtype)
        out = flat[offset : offset + size].view(shape)
        if form == "shares":
            ops.gemm_tiled_weight(x, wt, m, k, out, splits=5)
        else:
            ops.gemm_tiled_weight(x, wt, m, k, out, bias=bias, gated=form == "gated", accumulate=form == "added")
        assert bool((flat[:offset] == 5.0).all()) and bool((flat[offset + size :] == 5.0).all())
        return out

    out = run(0)
    assert torch.equal(out, run(4 if dtype == torch.bfloat16 else 2))  # eight bytes on
    got = out.double().sum(0) if form == "shares" else out.double()
    want = x.double() @ g.double().t()
    if form == "gated":
        want = want * torch.sigmoid(want) * (x.double() @ u.double().t())
    want += bias.double() if form == "bias" else 5.0 if form == "added" else 0.0
    # float32 sums of k products of numbers around k^-0.5, then at most one rounding to eight significant bits
    assert bool(((got - want).abs() <= (2.0**-8 if dtype == torch.bfloat16 else 0.0) * want.abs() + 1e-5 * k**0.5).all())
