"""Which float32 gate/up products apply the gate themselves: the sizes at which that is the faster way; the same bits either way."""

import pytest
import torch


@pytest.mark.parametrize("n, m, k, gated", [
    (4, 4864, 896, True), (509, 4864, 896, True), (1, 256, 1024, True), (1, 256, 1040, False), (16, 1024, 2048, False), (16, 1040, 2048, True),
    (1, 4096, 4096, True), (1, 4112, 4096, False), (8, 8192, 2048, False), (8, 8208, 2048, True), (8, 11264, 2048, True), (8, 11280, 2048, False),
    (17, 256, 512, True), (17, 256, 544, False), (256, 768, 2048, True), (128, 768, 2048, False), (17, 4112, 2048, True), (17, 4096, 2048, False),
    (32, 4112, 2048, True), (128, 768, 896, True), (96, 768, 896, False), (128, 768, 928, False), (509, 4864, 256, False), (4, 20, 64, False)])
def test_by_size(n, m, k, gated):
    from shrike_amd.kernels import ops

    assert ops.gemm_f32_gated_faster(n, m, k) is gated


class Step:
    def __init__(self):
        self.names = []

    def buffer(self, name, shape, dtype):
        self.names.append(name)
        return torch.empty(shape, dtype=dtype, device="cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("n, m, k", [(16, 1024, 1040), (16, 1040, 1040), (1, 48, 1024), (17, 64, 512), (17, 64, 544), (65, 2064, 1056), (130, 2064, 1056),
                                     (300, 1536, 1056), (509, 1536, 1056)])
def test_the_same_bits_whichever_way(n, m, k):
    from shrike_amd.engine.runtime import Runtime
    from shrike_amd.kernels import ops

    torch.manual_seed(n + m + k)
    runtime = Runtime(dtype=torch.float32)
    gate, up = (torch.randn(m, k, device="cuda") / k**0.5 for _ in range(2))
    w, x = runtime.gated_weight(gate, up, "gelu_tanh", 0.5, 1.0), torch.randn(n, k, device="cuda")
    step, out, both, want = Step(), torch.empty(n, m, device="cuda"), torch.empty(n, 2 * m, device="cuda"), torch.empty(n, m, device="cuda")
    runtime.gated_linear(step, x, w, out, "gelu_tanh", 0.5, 1.0)
    assert (step.names == []) is ops.gemm_f32_gated_faster(n, m, k)
    ops.gemm_f32_tiled_weight(x, w.tiled_f32, 2 * m, k, both)
    ops.act_mul(both, want, "gelu_tanh", 0.5, 1.0)
    assert torch.equal(out, want)
