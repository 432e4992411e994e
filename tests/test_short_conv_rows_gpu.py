"""The short convolution of many bfloat16 tokens in vectors against the general kernel, which takes rows that are not
aligned: the same sums in the same order, so the same bits."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("activation", [None, "silu"])
@pytest.mark.parametrize("before, starts", [
    ([], [0]),
    ([], [5]),  # inputs that the slot keeps
    ([1, 2, 3, 1, 7], [0, 1, 2, 3, 0, 9]),  # groups of several sequences, inputs before a sequence's start
    ([1] * 64, [40] * 64 + [1]),
])
@pytest.mark.parametrize("inner, more, last", [
    (2048, 24, 512),  # whole groups of tokens and whole workgroups
    (2056, 0, 513),  # a last group of one, a last workgroup of one thread
    (3584, 3584, 300), (10248, 0, 103)])
def test_rows_in_vectors_have_the_bits_of_the_general_kernel(inner, more, last, before, starts, activation):
    from shrike_amd.kernels import ops

    counts = [*before, last]
    torch.manual_seed(inner + len(counts))
    n, states = sum(counts), 1
    i32 = lambda values: torch.tensor(values, dtype=torch.int32, device="cuda")  # noqa: E731
    positions = i32([s + i for s, c in zip(starts, counts) for i in range(c)])
    token_seq = i32([q for q, c in enumerate(counts) for _ in range(c)])
    cu = i32([sum(counts[:q]) for q in range(len(counts) + 1)])
    slots = i32(torch.randperm(len(counts)).tolist())
    state = torch.randn(len(counts), inner * (states + 3), device="cuda")
    state[0, inner * states] = float("inf")  # (the oldest input of one sequence)
    taps, bias = torch.randn(inner, 4, device="cuda"), torch.randn(inner, device="cuda")
    x = torch.randn(n, inner + more, device="cuda").bfloat16()
    shifted = torch.empty(n, inner + more + 1, dtype=torch.bfloat16, device="cuda")
    shifted[:, 1:] = x
    got = []
    for rows in (x, shifted[:, 1:]):
        y = torch.full((n, inner), float("nan"), dtype=torch.bfloat16, device="cuda")
        ops.short_conv(rows, taps, bias, positions, token_seq, cu, slots, state, states, y, activation)
        got.append(y)
    assert torch.equal(got[0].view(torch.int16), got[1].view(torch.int16))
