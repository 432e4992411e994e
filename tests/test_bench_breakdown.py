"""bench.py's time of a step by kernel takes in every function that launches one (CPU)."""

import importlib.util
import inspect
import re
from pathlib import Path

from shrike_amd.csrc.build import CSRC
from shrike_amd.kernels import ops

spec = importlib.util.spec_from_file_location("bench", Path(__file__).resolve().parent.parent / "bench.py")
bench = importlib.util.module_from_spec(spec)
spec.loader.exec_module(bench)


def test_every_function_that_launches_a_kernel_is_timed():
    launchers = set(re.findall(r"SHK_LAUNCHER\((shk_\w+)\)", (CSRC / "calls.hip").read_text()))
    calling = {name for name, f in inspect.getmembers(ops, inspect.isfunction)
               if f.__module__ == ops.__name__ and launchers & set(re.findall(r"\.(shk_\w+)\(", inspect.getsource(f)))}
    # (what moves a step's metadata, or writes a slot's states outside of a step)
    aside = {"copy_words", "gather_rows", "zero_"}
    assert {"few_stream", "few_gated", "few_heads", "moe_few", "gemm_f32_groups", "gemm_f32_gated"} <= calling
    assert calling - aside == set(bench.TIMED_OPS)


def test_products_are_listed_by_their_matrix():
    class Out:
        shape = (8, 4608)

    assert bench.timed_label("few_stream", ("x", "w", 3584, 18944), {}) == "few_stream 3584x18944"
    assert bench.timed_label("few_heads", ("x", "w", 3584, Out), {}) == "few_heads 4608x3584"
    assert bench.timed_label("gemm_tiled_weight", ("x", "w", 37888, 3584), {"gated": "silu"}) == "gemm 37888x3584 gated"
    assert bench.timed_label("argmax", (), {}) == "argmax"
