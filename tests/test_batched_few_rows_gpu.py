"""Batches of products of few rows on both sides of the line between their kernels: what float64 gives, and the same bits as from the kernel that
serves outputs which are not 16-byte aligned."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch, n, m, k, dtype, lines", [
    (256, 1, 72, 128, torch.float32, True), (256, 8, 128, 128, torch.bfloat16, False), (256, 9, 72, 128, torch.bfloat16, True),
    (128, 12, 136, 192, torch.bfloat16, False), (128, 13, 136, 192, torch.bfloat16, True), (128, 3, 136, 192, torch.float32, True),
    (64, 16, 512, 512, torch.bfloat16, False), (64, 17, 512, 512, torch.bfloat16, True), (256, 48, 64, 64, torch.float32, False),
    (256, 49, 64, 64, torch.float32, True), (256, 17, 64, 128, torch.bfloat16, False), (256, 17, 64, 192, torch.bfloat16, True),
])
def test_few_rows(batch, n, m, k, dtype, lines):
    from shrike_amd.kernels import ops
    from tests.test_batched_lines_gpu import test_whole_lines

    assert ops.gemm_batched_lines(n, m, k, batch, dtype == torch.float32) == lines
    test_whole_lines(batch, n, m, k, dtype)
