"""The barrier between stages that are loaded straight into LDS: a wavefront has waited for its loads and for its
own reads of LDS before it meets the others, whose next loads overwrite what it read."""

import re
import subprocess

import pytest

from shrike_amd.csrc.build import CSRC, HIPCC_FLAGS, find_hipcc


def test_no_stage_is_freed_by_another_barrier():
    """In every source and header but the one that defines the loads and the barrier."""
    users = set()
    for path in sorted([*CSRC.glob("*.hip"), *CSRC.glob("*.h")]):
        if path.name == "to_lds.h":
            continue
        text = path.read_text()
        for name in ("__builtin_amdgcn_s_barrier", "__builtin_amdgcn_s_waitcnt", "__builtin_amdgcn_global_load_lds", "global_load_lds_dword",
                     "load_to_lds(", "s_barrier", "vmcnt"):
            assert name not in text, (path.name, name)
        if "SHK_LOAD_TO_LDS(" in text:
            users.add(path.name)
            assert "SHK_MEET_WITH_LOADS(" in text, path.name
    assert {"gemm_wide.h", "gemm_bf16.hip", "gemm_f32.hip", "attention_rows.hip"} <= users


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


def test_both_forms_of_the_load_in_one_kernel(tmp_path):
    """Each of three loads (builtin, base + offset, builtin) goes where it should: m0 is written anew before it; the barrier
    behind a load from base + offset waits for those before it and for reads of LDS."""
    hipcc = find_hipcc()
    if hipcc is None:
        pytest.skip("no hipcc")
    source = tmp_path / "both.hip"
    source.write_text("""
        #include "to_lds.h"
        __global__ void both(float* p) {
          __shared__ float a[256];
          const unsigned at = static_cast<unsigned>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)&a[0]));
          SHK_LOAD_TO_LDS(p + threadIdx.x * 4, a);
          SHK_LOAD_TO_LDS(at + 512u, threadIdx.x * 16u, reinterpret_cast<const char*>(p + 4096));
          SHK_LOAD_TO_LDS(p + 8192 + threadIdx.x * 4, a);
          SHK_MEET_WITH_LOADS(0);
          const float x = a[threadIdx.x ^ 1];
          SHK_LOAD_TO_LDS(at, threadIdx.x * 16u, reinterpret_cast<const char*>(p));
          SHK_LOAD_TO_LDS(at + 256u, threadIdx.x * 16u, reinterpret_cast<const char*>(p));
          SHK_MEET_WITH_LOADS(1);
          p[threadIdx.x] = a[threadIdx.x] + x;
        }
    """)
    out = tmp_path / "both.s"
    run = subprocess.run([hipcc, *HIPCC_FLAGS, f"-I{CSRC}", "--cuda-device-only", "-S", str(source), "-o", str(out)], check=True,
                         capture_output=True, text=True)
    assert "reserved register" not in run.stderr
    text = out.read_text()
    body = text[text.index("_Z4bothPf:") :]
    seen = re.findall(r"(m0, \S+)|(global_load_lds_dwordx4)", body[: body.index("s_endpgm")])
    places = []
    for place, load in seen:
        if place:
            last = place
        if load:
            places.append(last)
    assert places == ["m0, 0", "m0, 0x200", "m0, 0", "m0, 0", "m0, 0x100"]
    lines = [line.strip() for line in body[: body.index("s_endpgm")].splitlines()]
    lines = [line for line in lines if line and not line.startswith((";", "."))]
    waits = [lines[i - 1] for i, line in enumerate(lines) if line == "s_barrier"]
    assert [re.fullmatch(r"s_waitcnt vmcnt\((\d)\) lgkmcnt\(0\)", w).group(1) for w in waits] == ["0", "1"], waits
