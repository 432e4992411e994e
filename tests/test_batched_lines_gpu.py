"""Batches of products of many rows and whole stages of k: what float64 gives, and the same bits as from the kernel that serves outputs which are
not 16-byte aligned."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("batch, n, m, k", [(128, 129, 72, 64), (256, 17, 8, 128), (86, 257, 128, 448), (43, 383, 136, 192), (28, 641, 448, 128),
                                            (64, 128, 512, 256), (300, 1, 64, 64)])
def test_whole_lines(batch, n, m, k, dtype):
    from shrike_amd.kernels import ops

    torch.manual_seed(n + m)
    assert -(-n // 128) * -(-m // 128) * batch >= 256
    a = torch.randn(n, batch * k, device="cuda").bfloat16()
    w = (torch.randn(batch, m, k, device="cuda") / k**0.5).bfloat16()

    def run(offset):
        flat = torch.full((n * batch * m + 8,), 5.0, device="cuda", dtype=dtype)
        out = flat[offset : offset + n * batch * m].view(n, batch * m)
        ops.gemm_batched(a, w, out, batch, k, m)
        assert bool((flat[:offset] == 5.0).all()) and bool((flat[offset + n * batch * m :] == 5.0).all())
        return out

    out = run(0)
    assert torch.equal(out, run(2 if dtype == torch.float32 else 4))  # eight bytes on
    want = torch.bmm(a.view(n, batch, k).transpose(0, 1).contiguous().double(), w.double().transpose(1, 2).contiguous())
    want = want.transpose(0, 1).reshape(n, -1)
    # float32 sums of k products of numbers around k^-0.5, then at most one rounding to eight significant bits
    assert bool(((out.double() - want).abs() <= (0.0 if dtype == torch.float32 else 2.0**-8) * want.abs() + 1e-5 * k**0.5).all())
