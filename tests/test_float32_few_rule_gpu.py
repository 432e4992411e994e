"""Which float32 products of up to 16 rows run in the kernel for few of them: the sizes that it serves faster; the same bits on both
sides of each line."""

import pytest
import torch


@pytest.mark.parametrize("n, m, k, few", [
    (4, 896, 896, True), (16, 2048, 2560, True), (16, 2048, 2576, False), (1, 256, 8192, False), (16, 2064, 2576, True), (16, 8192, 14336, True),
    (4, 9728, 896, True), (16, 12288, 1024, True), (1, 8208, 1040, False), (1, 11008, 2048, False), (4, 32000, 2048, False),
    (4, 151936, 896, True), (9, 151936, 896, False), (4, 50000, 256, False), (8, 16384, 1024, True), (8, 16384, 1040, False),
    (17, 896, 896, False), (4, 896, 900, False)])
def test_by_size(n, m, k, few):
    from shrike_amd.kernels import ops

    assert ops.gemm_f32_few(n, m, k) is few


@pytest.mark.gpu
@pytest.mark.parametrize("m, k", [(40, 2560), (40, 2576), (2048, 2560), (2048, 2576), (2050, 2576), (8192, 1040), (8194, 1024), (8194, 1040), (12290, 896),
                                  (12290, 1040)])
def test_the_same_bits_on_both_sides(m, k):
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k)
    a, wt = torch.randn(16, k + 1, device="cuda"), ops.retile_f32(torch.randn(m, k, device="cuda") / k**0.5)
    rows = a[:, 1:].contiguous()
    want = torch.empty(16, m, device="cuda")
    ops.gemm_f32_tiled_weight(a[:, 1:], wt, m, k, want)  # (rows that are not aligned: the general kernel)
    for n in (1, 8, 9, 16):
        out = torch.empty(n, m, device="cuda")
        ops.gemm_f32_tiled_weight(rows[:n], wt, m, k, out)
        assert torch.equal(out, want[:n])
