"""Float32 products on the matrix units: against float64 at the edges of every tile shape, and the same
bits for a row whatever shape the number of rows selects, tiled weights or not."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from shrike_amd.kernels import ops

    return ops


# k: one element, a step and one more, a segment's edge, many steps a segment; m and n around 16, 32 and 64
@pytest.mark.parametrize("m, k", [(1, 1), (17, 16), (64, 17), (130, 70), (896, 896), (2052, 257), (333, 4864), (33000, 40)])
@pytest.mark.parametrize("aligned", [True, False])
def test_against_float64_and_the_same_bits_for_any_number_of_rows(ops, m, k, aligned):
    torch.manual_seed(m + k)
    n_max = 70 if m > 20000 else 1100 if m == 896 else 260
    wide = torch.randn(n_max, k + 5, device="cuda")
    a = wide[:, :k] if not aligned else wide[:, :k].contiguous()
    w, bias = torch.randn(m, k, device="cuda"), torch.randn(m, device="cuda")
    wt = ops.retile_f32(w)
    full = None
    for n in [n_max, 1, 2, 15, 16, 17, 31, 33, 64, 65, 129]:
        if n > n_max:
            continue
        rows, tiled = torch.full((n, m + 3), 7.0, device="cuda"), torch.full((n, m), 7.0, device="cuda")
        ops.gemm(a[:n], w, rows[:, :m], bias=bias)
        ops.gemm_f32_tiled_weight(a[:n], wt, m, k, tiled, bias=bias)
        assert bool((rows[:, m:] == 7.0).all())
        assert torch.equal(rows[:, :m], tiled)
        if full is None:
            full = tiled
            exact = a.double() @ w.double().t() + bias.double()
            # at most k / 16 + 40 roundings on the way of a product into its sum, each of half an ulp of a partial
            # sum that the sum of the products' sizes bounds
            size = a.double().abs() @ w.double().abs().t() + bias.double().abs()
            assert bool(((tiled.double() - exact).abs() <= (k / 16 + 40) * 2.0**-24 * size).all())
        assert torch.equal(tiled, full[:n])
        again = tiled.clone()
        ops.gemm_f32_tiled_weight(a[:n], wt, m, k, again, accumulate=True)
        plain = torch.empty_like(tiled)
        ops.gemm_f32_tiled_weight(a[:n], wt, m, k, plain)
        assert torch.equal(again, plain + tiled)


@pytest.mark.parametrize("batch, m, k", [(28, 448, 128), (14, 128, 64), (40, 250, 192), (16, 96, 77), (3, 900, 256), (5, 512, 260), (9, 700, 16)])
def test_many_rows_of_a_short_k_in_batches(ops, batch, m, k):
    torch.manual_seed(batch + k)
    n_max = 700
    a, w = torch.randn(n_max, batch * k, device="cuda"), torch.randn(batch, m, k, device="cuda")
    per = a.view(n_max, batch, k).transpose(0, 1).double()
    exact = torch.stack([per[b] @ w[b].double().t() for b in range(batch)], 1).view(n_max, batch * m)
    size = torch.stack([per[b].abs() @ w[b].double().abs().t() for b in range(batch)], 1).view(n_max, batch * m)
    full = None
    for n in (n_max, 1, 17, 100, 300, 511):
        out = torch.full((n, batch * m + 4), 7.0, device="cuda")
        ops.gemm_batched(a[:n], w, out[:, : batch * m], batch, k, m)
        assert bool((out[:, batch * m :] == 7.0).all())
        full = out if full is None else full
        assert torch.equal(out, full[:n]), "the same bits in every shape"
    assert bool(((full[:, : batch * m].double() - exact).abs() <= (k / 16 + 40) * 2.0**-24 * size).all())


def test_what_does_not_fit_is_refused(ops):
    from shrike_amd.kernels import KernelError

    a, wt = torch.zeros(2, 8, device="cuda"), ops.retile_f32(torch.zeros(4, 8, device="cuda"))
    with pytest.raises(KernelError, match="tiled weights"):
        ops.gemm_f32_tiled_weight(a, wt, 17, 8, torch.zeros(2, 17, device="cuda"))
    with pytest.raises(KernelError):
        ops.gemm_f32_tiled_weight(a, wt, 4, 8, torch.zeros(2, 5, device="cuda"))
    with pytest.raises(KernelError):
        ops.retile_f32(torch.zeros(4, 8, device="cuda", dtype=torch.bfloat16))
