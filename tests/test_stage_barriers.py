"""The barrier between stages that are loaded straight into LDS: a wavefront has waited for its loads and for its
own reads of LDS before it meets the others, whose next loads overwrite what it read."""

import re
import subprocess

import pytest

from shrike_amd.csrc.build import CSRC, HIPCC_FLAGS, find_hipcc


def test_no_stage_is_freed_by_another_barrier():
    users = 0
    for path in sorted(CSRC.glob("*.hip")):
        text = path.read_text()
        assert "__builtin_amdgcn_s_barrier" not in text and "__builtin_amdgcn_s_waitcnt" not in text, path.name
        if "SHK_LOAD_TO_LDS(" in text:
            users += 1
            assert "SHK_MEET_WITH_LOADS(" in text, path.name
    assert users >= 2


def test_the_barrier_waits_for_reads_of_lds(tmp_path):
    hipcc = find_hipcc()
    if hipcc is None:
        pytest.skip("no hipcc")
    source = tmp_path / "meet.hip"
    source.write_text("""
        #include "to_lds.h"
        template <int N>
        __global__ void meet(float* p) {
          __shared__ float a[64];
          SHK_LOAD_TO_LDS(p + threadIdx.x * 4, a);
          SHK_MEET_WITH_LOADS(N);
          const float x = a[threadIdx.x ^ 1];
          SHK_MEET_WITH_LOADS(0);
          a[threadIdx.x] = x * 2.f;
          SHK_WAIT_LOADS(N);
          p[threadIdx.x] = a[threadIdx.x];
        }
        template __global__ void meet<6>(float*);
        template __global__ void meet<23>(float*);
    """)
    out = tmp_path / "meet.s"
    subprocess.run([hipcc, *HIPCC_FLAGS, f"-I{CSRC}", "--cuda-device-only", "-S", str(source), "-o", str(out)], check=True,
                   capture_output=True)
    text = out.read_text()
    for n in (6, 23):
        body = text[text.index(f"_Z4meetILi{n}EEvPf:") :]
        lines = [line.strip() for line in body[: body.index("s_endpgm")].splitlines()]
        lines = [line for line in lines if line and not line.startswith((";", "."))]
        barriers = [i for i, line in enumerate(lines) if line == "s_barrier"]
        assert len(barriers) == 2
        for i, count in zip(barriers, (n, 0)):
            assert re.fullmatch(rf"s_waitcnt vmcnt\({count}\) lgkmcnt\(0\)", lines[i - 1]), lines[i - 1]
        assert f"s_waitcnt vmcnt({n})" in lines[barriers[1] :]  # (the wait alone leaves reads of LDS in flight)
