"""Products of few tokens that add to the stream, in half blocks of weight rows: a row's bits are those of the same row in a matrix that
runs in whole blocks, and of the same token among others."""

import pytest
import torch

pytestmark = pytest.mark.gpu

WIDE = 3072  # rows of a matrix that runs in whole blocks, whatever k


def run(ops, w, a, before, weight, bias):
    (m, k), n = w.shape, a.shape[0]
    resid = before[:, :m].clone(memory_format=torch.contiguous_format)
    rows = torch.empty(m // 8, n, 8, device="cuda", dtype=torch.bfloat16)
    sums = torch.full((ops.few_stream_sums(n, m, k), n), float("nan"), device="cuda")
    ops.few_stream(a, ops.retile_weight(w), m, k, resid, weight[:m].contiguous(), rows, sums, bias=bias[:m].contiguous())
    return resid, rows.transpose(0, 1).reshape(n, m), sums


# one k-tile; an odd number of them, the last one whole or not; wavefronts' walks of one tile up to ten, asked for at once; longer ones in
# batches, one to four of them; walks in even and odd numbers
@pytest.mark.parametrize("m, k", [(16, 8), (896, 896), (1008, 328), (1024, 1056), (512, 1600), (1536, 2568), (896, 4864), (1024, 4104),
                                  (1536, 6144), (2048, 5144), (2048, 8192)])
def test_half_blocks_give_the_bits_of_whole_ones(m, k):
    from shrike_amd.kernels import ops

    torch.manual_seed(m + k)
    a = torch.randn(64, k, device="cuda").bfloat16()
    w = (torch.randn(WIDE, k, device="cuda") / k**0.5).bfloat16()
    weight, bias, before = 1 + 0.1 * torch.randn(WIDE, device="cuda"), torch.randn(WIDE, device="cuda"), torch.randn(64, WIDE, device="cuda")
    assert ops.few_stream_sums(16, m, k) == m // 8 and ops.few_stream_sums(16, WIDE, k) == WIDE // 16
    whole = [torch.cat(x) for x in zip(*(run(ops, w, a[i : i + 16], before[i : i + 16], weight, bias)[:2] for i in range(0, 64, 16)))]
    for n in (1, 7, 8, 9, 15, 16, 17, 24, 32, 33, 64):
        if ops.few_stream_sums(n, m, k) == 0:
            assert n > 16 and m * k > 5_000_000
            continue
        resid, rows, sums = run(ops, w[:m], a[64 - n :], before[64 - n :], weight, bias)
        assert torch.equal(resid, whole[0][64 - n :, :m]) and torch.equal(rows, whole[1][64 - n :, :m]), n
        squares = (resid.double() ** 2).view(n, m // 8, 8).sum(-1).t()
        assert bool(((sums.double() - squares).abs() <= 8 * 2.0**-24 * squares).all()), n
    exact = before[:, :m].double() + a.double() @ w[:m].double().t() + bias[:m].double()
    size = before[:, :m].double().abs() + a.double().abs() @ w[:m].double().abs().t() + bias[:m].double().abs()
    # a float32 sum over k: a rounding a step of 32, whose own order is the matrix unit's (40 more), then stream and bias
    assert bool(((whole[0][:, :m].double() - exact).abs() <= ((k / 32 + 40) * 2.0**-24 + 2.0**-22) * size).all())
