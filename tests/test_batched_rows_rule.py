"""Which batches of products take the kernel whose workgroups form 128 rows and features each: where they fill the compute units, but few rows only
where it is the faster one all the same."""

import pytest

from shrike_amd.kernels import ops


@pytest.mark.parametrize("batch, k, m, f32, first", [
    (256, 64, 128, False, 49), (256, 64, 128, True, 49), (300, 64, 64, False, 49), (64, 64, 512, True, 49),  # one stage of k
    (256, 128, 64, False, 49), (256, 192, 64, True, 17), (256, 512, 64, False, 17),                          # half the features idle
    (64, 128, 512, False, 9), (64, 128, 512, True, 1), (256, 192, 72, False, 13), (128, 192, 256, True, 1),
    (64, 512, 512, False, 17), (64, 512, 512, True, 17), (128, 256, 256, False, 17), (256, 4096, 128, True, 17),
])
def test_few_rows_keep_the_kernel_for_them(batch, k, m, f32, first):
    assert [n for n in range(1, 129) if ops.gemm_batched_lines(n, m, k, batch, f32)] == list(range(first, 129))


def test_not_where_its_workgroups_leave_compute_units_idle():
    assert not ops.gemm_batched_lines(100, 128, 128, 255) and ops.gemm_batched_lines(129, 128, 128, 128)
    assert not ops.gemm_batched_lines(1000, 448, 100, 28) and ops.gemm_batched_lines(1000, 448, 128, 28)  # k in whole stages
    # latent attention: single tokens of 64 and 128 heads of 128 elements over 512 latent features
    assert not ops.gemm_batched_lines(8, 512, 128, 64) and not ops.gemm_batched_lines(1, 128, 512, 128)
