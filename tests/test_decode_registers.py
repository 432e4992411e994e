"""Decode attention for heads of 128 elements: registers for two workgroups of four wavefronts on a compute unit (512 a lane and SIMD), without
scratch memory.  With one workgroup a compute unit 256 sequences of 300 keys take 12 to 15 % longer."""

import re
import subprocess

import pytest

from shrike_amd.csrc.build import CSRC, FILE_FLAGS, HIPCC_FLAGS, find_hipcc


def test_two_workgroups_share_a_compute_unit(tmp_path):
    hipcc = find_hipcc()
    if hipcc is None:
        pytest.skip("no hipcc")
    out = tmp_path / "attention.s"
    subprocess.run([hipcc, *HIPCC_FLAGS, *FILE_FLAGS["attention_mfma.hip"], "--cuda-device-only", "-S", str(CSRC / "attention_mfma.hip"),
                    "-o", str(out)], check=True, capture_output=True)
    kernels = re.findall(r"\.name: +(\S+)\n(.*?)\n +\.wavefront_size", out.read_text(), re.S)
    seen = [(name, dict(re.findall(r"\.(\w+): +(\d+)", body))) for name, body in kernels if "attention_decode_kernelILi128E" in name]
    assert len(seen) >= 4  # with and without non-temporal loads, pages of 16 and of any size
    for name, of in seen:
        assert int(of["vgpr_count"]) <= 256, (name, of["vgpr_count"])  # (accumulation registers among them)
        assert int(of["private_segment_fixed_size"]) == 0 and int(of["vgpr_spill_count"]) == 0, name
