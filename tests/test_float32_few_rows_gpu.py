"""float32 products of up to 16 rows: the bits of the same rows among more of them, whole, in groups and with the gate,
at the edges of segments, batches of steps and blocks of features; groups and gate of more rows against the whole product."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(16, 16), (40, 256), (896, 896), (1152, 912), (37, 2576), (896, 4864), (2064, 1024), (3584, 1040), (2080, 4880)]


def operands(m, k):
    torch.manual_seed(m + k)
    a = torch.randn(33, k, device="cuda")
    return a, torch.randn(m, k, device="cuda") / k**0.5


@pytest.mark.parametrize("n", [1, 4, 15, 16])
@pytest.mark.parametrize("m, k", SIZES)
def test_the_same_bits_as_among_more_rows(m, k, n):
    from shrike_amd.kernels import ops

    a, w = operands(m, k)
    wt, bias = ops.retile_f32(w), torch.randn(m, device="cuda")
    whole = torch.empty(33, m, device="cuda")
    ops.gemm_f32_tiled_weight(a, wt, m, k, whole, bias=bias)
    out = torch.full((n, m + 4), 7.0, device="cuda")
    ops.gemm_f32_tiled_weight(a[5 : 5 + n], wt, m, k, out[:, :m], bias=bias)
    assert torch.equal(out[:, :m], whole[5 : 5 + n]) and bool((out[:, m:] == 7.0).all())
    ops.gemm_f32_tiled_weight(a[5 : 5 + n], wt, m, k, out[:, :m], bias=bias, accumulate=True)
    assert torch.equal(out[:, :m], whole[5 : 5 + n] + whole[5 : 5 + n])
    exact = a.double() @ w.double().t() + bias.double()
    size = a.double().abs() @ w.double().abs().t() + bias.double().abs()
    # a sum over k in 16 segments of steps, four groups, the bias: a rounding each
    assert bool(((whole.double() - exact).abs() <= (k / 16 + 24) * 2.0**-24 * size).all())


@pytest.mark.parametrize("n", [1, 5, 16])
@pytest.mark.parametrize("m, k", [(896, 4864), (1536, 8960), (20, 2048), (2048, 2064)])
def test_groups_that_the_norm_adds(m, k, n):
    from shrike_amd.kernels import ops

    assert ops.gemm_f32_splits(n, m, k) == 4 and ops.gemm_f32_splits(17, m, k) == 1
    a, w = operands(m, k)
    wt = ops.retile_f32(w)
    whole, parts = torch.empty(n, m, device="cuda"), torch.empty(4, n, m, device="cuda")
    ops.gemm_f32_tiled_weight(a[:n], wt, m, k, whole)
    ops.gemm_f32_groups(a[:n], wt, m, k, parts)
    assert torch.equal(((parts[0] + parts[1]) + parts[2]) + parts[3], whole)
    resid, weight = torch.randn(n, m, device="cuda"), torch.randn(m, device="cuda")
    results = []
    for delta in (whole, ops.SplitSum(parts)):
        x, out = resid.clone(), torch.empty(n, m, device="cuda")
        ops.add_rmsnorm(x, delta, weight, 1e-6, out)
        results.append((x, out))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.parametrize("n", [1, 7, 16])
@pytest.mark.parametrize("m, k", [(16, 16), (48, 512), (4864, 896), (304, 1024), (320, 1040), (64, 4880)])
@pytest.mark.parametrize("activation, limit, shift", [("silu", None, 0.0), ("gelu_tanh", 0.5, 1.0), ("relu", None, 0.0), ("quick_gelu", 0.7, 0.0)])
def test_a_gate_in_the_product(m, k, n, activation, limit, shift):
    from shrike_amd.kernels import ops

    assert ops.gemm_f32_gated_takes(n, m, k)
    a, w = operands(2 * m, k)
    wt = ops.retile_f32(w)
    both, want = torch.empty(n, 2 * m, device="cuda"), torch.empty(n, m, device="cuda")
    ops.gemm_f32_tiled_weight(a[:n], wt, 2 * m, k, both)
    ops.act_mul(both, want, activation, limit, shift)
    out = torch.empty(n, m, device="cuda")
    ops.gemm_f32_gated(a[:n], wt, m, k, out, activation, limit, shift)
    assert torch.equal(out, want)


@pytest.mark.parametrize("n", [64, 65, 200, 509])
@pytest.mark.parametrize("m, k", [(896, 4864), (20, 4096), (1004, 4128), (64, 8992)])
def test_groups_of_more_rows(m, k, n):
    from shrike_amd.kernels import ops

    assert ops.gemm_f32_splits(n, m, k) == 4 and ops.gemm_f32_splits(2000, 896, 4864) == ops.gemm_f32_splits(n, m, k + 16) == 1
    torch.manual_seed(m + k + n)
    a, w = torch.randn(n, k + 4, device="cuda")[:, :k], torch.randn(m, k, device="cuda") / k**0.5
    wt, whole, parts = ops.retile_f32(w), torch.empty(n, m, device="cuda"), torch.full((4, n, m), 7.0, device="cuda")
    ops.gemm_f32_tiled_weight(a, wt, m, k, whole)
    ops.gemm_f32_groups(a, wt, m, k, parts)
    assert torch.equal(((parts[0] + parts[1]) + parts[2]) + parts[3], whole)


@pytest.mark.parametrize("n", [17, 32, 33, 64, 65, 509])
@pytest.mark.parametrize("m, k", [(16, 288), (48, 512), (4864, 896), (304, 1056), (64, 4896)])
def test_a_gate_in_the_product_of_more_rows(m, k, n):
    from shrike_amd.kernels import ops

    assert ops.gemm_f32_gated_takes(n, m, k) and not ops.gemm_f32_gated_takes(n, m, 256)
    torch.manual_seed(m + k + n)
    a, w = torch.randn(n, k + 4, device="cuda")[:, :k], torch.randn(2 * m, k, device="cuda") / k**0.5
    wt = ops.retile_f32(w)
    both, want, out = torch.empty(n, 2 * m, device="cuda"), torch.empty(n, m, device="cuda"), torch.empty(n, m, device="cuda")
    ops.gemm_f32_tiled_weight(a, wt, 2 * m, k, both)
    ops.act_mul(both, want, "gelu_tanh", 0.5, 1.0)
    ops.gemm_f32_gated(a, wt, m, k, out, "gelu_tanh", 0.5, 1.0)
    assert torch.equal(out, want)
