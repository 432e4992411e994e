"""Which products of few tokens go the way of gemm_few.hip: the sizes at which it is the faster one, alike for every number of tokens that a
recorded step stands for (CPU)."""

import pytest

from shrike_amd.kernels import ops


@pytest.mark.parametrize("n, m, k, stream", [
    (1, 896, 4864, True), (8, 3584, 18944, True), (16, 3584, 3584, True), (64, 896, 896, True), (64, 896, 4864, True),
    (1, 512, 5120, True), (1, 512, 5128, False), (1, 1536, 6144, True), (8, 1536, 8960, False), (1, 2048, 8192, True), (1, 2048, 8200, False),
    (8, 2560, 8960, True), (8, 2560, 8968, False), (16, 3072, 24576, True), (64, 256, 5120, True), (64, 256, 6144, False), (8, 5120, 5120, False)])
def test_products_that_add_to_the_stream(n, m, k, stream):
    assert (ops.few_stream_sums(n, m, k) > 0) is stream


@pytest.mark.parametrize("n, m, k, heads", [
    (16, 10240, 8192, True), (17, 2560, 2048, True), (32, 4096, 2304, True), (32, 4096, 2560, False), (17, 6144, 2048, False), (32, 4608, 2304, False),
    (33, 2560, 2304, True), (33, 4096, 2304, False), (65, 2048, 1536, True), (128, 1152, 896, True), (512, 1152, 896, False), (513, 768, 256, False)])
def test_projections_to_heads(n, m, k, heads):
    assert ops.few_heads_takes(n, m, k) is heads


@pytest.mark.parametrize("m, k", [(896, 896), (1152, 896), (896, 4864), (3584, 3584), (3584, 18944), (2048, 2048), (6144, 2048), (4096, 2304), (1536, 512)])
def test_alike_for_every_row_count_of_a_graph_bucket(m, k):
    for lo, hi in ((1, 16), (17, 32), (33, 64), (65, 128), (129, 256)):
        plans = {(ops.few_stream_sums(n, m, k) if n <= 64 else 0, ops.few_gated_takes(n, m, k) if n <= 64 else False, ops.few_heads_takes(n, m, k))
                 for n in range(lo, hi + 1)}
        assert len(plans) == 1, f"rows {lo}..{hi} of [{m}, {k}]: {sorted(plans)}"
