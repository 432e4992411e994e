"""Which float32 products leave groups of k for the norm that follows: the sizes at which both are done sooner so."""

import pytest
import torch


@pytest.mark.parametrize("n, m, k, groups", [
    (4, 896, 4864, True), (16, 1024, 2560, True), (1, 1024, 2576, False), (16, 1024, 4096, True), (9, 1028, 4096, False), (8, 1028, 4096, True),
    (16, 1536, 2560, True), (1, 1540, 2560, False), (4, 2048, 5632, False), (4, 1536, 8960, True), (16, 1536, 8960, False), (4, 896, 896, False),
    (509, 896, 4864, True), (100, 896, 4864, True), (64, 896, 4864, False), (256, 256, 4096, False), (257, 256, 4096, True), (2000, 896, 4864, False)])
def test_by_size(n, m, k, groups):
    from shrike_amd.kernels import ops

    assert ops.gemm_f32_groups_faster(n, m, k) is groups


@pytest.mark.gpu
@pytest.mark.parametrize("n, m, k", [(4, 896, 4864), (16, 1028, 4096), (64, 256, 4096), (257, 256, 4096)])
def test_a_sublayers_last_product_joins_with_the_same_bits(n, m, k):
    from types import SimpleNamespace

    from shrike_amd.engine.runtime import Runtime
    from shrike_amd.kernels import ops

    torch.manual_seed(n + m)
    runtime = Runtime(dtype=torch.float32)
    w, x = runtime.weight(torch.randn(m, k, device="cuda") / k**0.5), torch.randn(n, k, device="cuda")
    weight, results = torch.randn(m, device="cuda"), []
    for onto in (None, (None, None, False)):  # (nothing said about the stream; a norm that takes parts comes next)
        step = SimpleNamespace(onto=onto, num_tokens=n, buffer=lambda name, shape, dtype: torch.empty(shape, dtype=dtype, device="cuda"))
        delta = runtime.linear_onto(step, "out", x, w)
        assert isinstance(delta, ops.SplitSum) is (onto is not None and ops.gemm_f32_groups_faster(n, m, k)) and step.onto is None
        resid, out = torch.ones(n, m, device="cuda"), torch.empty(n, m, device="cuda")
        ops.add_rmsnorm(resid, delta, weight, 1e-6, out)
        results.append((resid, out))
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("n, m, k", [(3, 20, 16), (16, 24, 272), (5, 40, 1024), (16, 24, 2560), (16, 24, 2576)])
def test_groups_of_any_k(n, m, k):
    from shrike_amd.kernels import ops

    torch.manual_seed(n + k)
    a, wt = torch.randn(n, k, device="cuda"), ops.retile_f32(torch.randn(m, k, device="cuda") / k**0.5)
    whole, parts = torch.empty(n, m, device="cuda"), torch.full((4, n, m), 7.0, device="cuda")
    ops.gemm_f32_tiled_weight(a, wt, m, k, whole)
    ops.gemm_f32_groups(a, wt, m, k, parts)
    assert torch.equal(((parts[0] + parts[1]) + parts[2]) + parts[3], whole)
