"""Latent attention of single tokens in the prompt portions' kernel: few columns a workgroup, rows in many shares, against the
kernel for single tokens, and the shares that a step's shape gives."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads, key_dim, v_dim, page", [(28, 512, 448, 16), (32, 512, 130, 16), (33, 512, 512, 32), (14, 176, 112, 16),
                                                         (16, 256, 256, 64), (4, 40, 24, 4)])
@pytest.mark.parametrize("nsplit", [1, 2, 9, 64])
def test_the_same_as_the_kernel_for_single_tokens(heads, key_dim, v_dim, page, nsplit):
    from shrike_amd.kernels import ops

    torch.manual_seed(heads + key_dim)
    ctx = [1, 31, 32, 33, 64, 257, 850]
    n, per = len(ctx), -(-max(ctx) // page)
    pool = torch.full((n * per, page, key_dim), float("nan"), device="cuda", dtype=torch.bfloat16)
    tables = torch.randperm(n * per, device="cuda").view(n, per).int()
    for s, c in enumerate(ctx):
        at = torch.arange(c, device="cuda")
        pool[tables[s].long()[at // page], at % page] = torch.randn(c, key_dim, device="cuda").bfloat16()
    q = torch.randn(n, heads * key_dim, device="cuda").bfloat16()
    positions = torch.tensor([c - 1 for c in ctx], dtype=torch.int32, device="cuda")
    seqs = torch.arange(n, dtype=torch.int32, device="cuda")
    outs = []
    for kernel, more in ((ops.latent_attention_mfma, {}), (ops.latent_prompt, {"tokens": 1})):
        out = torch.full((n, heads * v_dim), float("nan"), device="cuda", dtype=torch.bfloat16)
        partial = torch.full((n * heads * nsplit * (v_dim + 2),), float("nan"), device="cuda")
        kernel(q, out, heads, key_dim, v_dim, positions, seqs, tables, pool, page, None, 0.7 / key_dim**0.5, partial=partial, nsplit=nsplit,
               **more)
        outs.append(out)
    assert torch.equal(*outs) and bool(torch.isfinite(outs[0].float()).all())
    # one key: its value
    assert torch.equal(outs[0][0].view(heads, v_dim), pool[tables[0, 0].long(), 0, :v_dim].expand(heads, v_dim))
