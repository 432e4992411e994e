"""The gated float32 product into rows that do not begin at a multiple of 16 bytes: the bits of aligned ones, and nothing beside them."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 16, 17, 33, 509])
@pytest.mark.parametrize("m, k", [(16, 288), (304, 1056), (4864, 896)])
@pytest.mark.parametrize("offset", [1, 2, 3])
def test_rows_at_any_element(m, k, n, offset):
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k + n)
    a, wt = torch.randn(n, k, device="cuda"), ops.retile_f32(torch.randn(2 * m, k, device="cuda") / k**0.5)
    want, room = torch.empty(n, m, device="cuda"), torch.full((n * m + 8,), 7.0, device="cuda")
    ops.gemm_f32_gated(a, wt, m, k, want, "silu")
    out = room[offset : offset + n * m].view(n, m)
    assert out.data_ptr() % 16 == 4 * offset
    ops.gemm_f32_gated(a, wt, m, k, out, "silu")
    assert torch.equal(out, want)
    assert bool((room[:offset] == 7.0).all()) and bool((room[offset + n * m :] == 7.0).all())
