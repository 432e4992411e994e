"""The short convolution of many short sequences: in vectors only where sequences are long enough for it, and with the general kernel's
bits where many of a step's inputs come from the slots."""

import pytest
import torch


@pytest.mark.parametrize("n, inner, seqs, vectors", [
    (1501, 3584, 1, True), (512, 3584, 1, True), (512, 2048, 1, True), (511, 2048, 1, False),
    (600, 3584, 600, False), (600, 3584, 150, False), (600, 3584, 120, True), (2048, 896, 512, False), (2048, 896, 400, True),
    (600, 2048, 25, False), (640, 2048, 10, True), (2048, 3584, 2048, False), (2048, 3584, 1024, True)])
def test_which_steps_move_vectors(n, inner, seqs, vectors):
    from shrike_amd.kernels import ops

    assert ops.short_conv_in_vectors(n, inner, seqs) is vectors


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[2] * 1024, [5] * 200 + [3, 1] + [7] * 150, [1] * 300 + [1701]])
def test_the_bits_of_the_general_kernel(counts):
    from shrike_amd.kernels import ops

    inner, states, n = 2056, 1, sum(counts)
    assert ops.short_conv_in_vectors(n, inner, len(counts))
    torch.manual_seed(n)
    i32 = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")  # noqa: E731
    starts = [q % 5 for q in range(len(counts))]
    positions = i32([s + i for s, c in zip(starts, counts) for i in range(c)])
    token_seq = i32([q for q, c in enumerate(counts) for _ in range(c)])
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), torch.cumsum(torch.tensor(counts), 0)]).int().cuda()
    slots = torch.randperm(len(counts)).int().cuda()
    state = torch.randn(len(counts), inner * (states + 3), device="cuda")
    taps, bias = torch.randn(inner, 4, device="cuda"), torch.randn(inner, device="cuda")
    x = torch.randn(n, inner, device="cuda").bfloat16()
    shifted = torch.empty(n, inner + 1, dtype=torch.bfloat16, device="cuda")
    shifted[:, 1:] = x
    got = []
    for rows in (x, shifted[:, 1:]):
        y = torch.full((n, inner), float("nan"), dtype=torch.bfloat16, device="cuda")
        ops.short_conv(rows, taps, bias, positions, token_seq, cu, slots, state, states, y, "silu")
        got.append(y)
    assert torch.equal(got[0].view(torch.int16), got[1].view(torch.int16))
