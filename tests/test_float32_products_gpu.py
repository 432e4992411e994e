"""float32 products of many rows whose operands are shared through LDS: the bits of the other shapes of the kernel, at the
edges of tiles, segments and rings."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, m, k", [(509, 9728, 896), (64, 9728, 288), (300, 896, 1024), (2000, 1152, 320), (33, 9000, 512), (513, 2056, 2048),
                                     (1024, 897, 1056), (1501, 3590, 352), (290, 1001, 992)])
def test_every_row_has_the_bits_that_few_rows_have(n, m, k):
    from shrike_amd.kernels import ops

    gen = torch.Generator("cuda").manual_seed(n + m + k)
    x = torch.randn(n, k, generator=gen, device="cuda")
    w = torch.randn(m, k, generator=gen, device="cuda") / k**0.5
    bias = torch.randn(m, generator=gen, device="cuda")
    wt = ops.retile_f32(w)
    out = torch.full((n, m), float("nan"), device="cuda")
    ops.gemm_f32_tiled_weight(x, wt, m, k, out)
    want = x.double() @ w.double().T
    # sums of k products in float32: at most k 2^-24 of the sum of magnitudes, some sqrt(k) of a result's size
    assert (out.double() - want).abs().max() < k * 2.0**-24 * want.abs().max()
    for first in sorted({0, 17, n // 2, n - 7}):
        few = torch.empty(7, m, device="cuda")
        ops.gemm_f32_tiled_weight(x[first : first + 7], wt, m, k, few)
        assert torch.equal(few, out[first : first + 7])
    # rows of wider buffers, what lies beyond them infinite; a bias; added to what is there
    apart = torch.full((n, k + 8), float("inf"), device="cuda")
    apart[:, :k] = x
    wide = torch.full((n, m + 3), 2.0, device="cuda")
    ops.gemm_f32_tiled_weight(apart[:, :k], wt, m, k, wide[:, :m], bias=bias)
    assert torch.equal(wide[:, :m], out + bias) and (wide[:, m:] == 2.0).all()
    ops.gemm_f32_tiled_weight(x, wt, m, k, wide[:, :m], accumulate=True)
    assert torch.equal(wide[:, :m], (out + bias) + out)
