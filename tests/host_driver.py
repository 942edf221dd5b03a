"""The path a multi-token attention call takes, from the library's own plan
(llmplayer_amd/csrc/prefill_plan.h through tests/host_layout_check.cpp, built with g++ once per run)."""
import functools
import os
import shutil
import subprocess
import tempfile

import pytest

from llmplayer_amd import hip_forward_pass as hfp

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@functools.lru_cache(maxsize=None)
def _driver():
    if shutil.which("g++") is None:
        pytest.skip("needs g++ for the plan of a call")
    exe = os.path.join(tempfile.mkdtemp(), "host_layout_check")
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", os.path.join(ROOT, "llmplayer_amd", "csrc"), "-I",
                    os.path.join(ROOT, "include"), os.path.join(ROOT, "tests", "host_layout_check.cpp"), "-o", exe],
                   check=True)
    return exe


def wide_form(c, layer, pos0, n):
    """"" for a call on the 16x16 path, else the wide attention's launch form: "one" block per
    workgroup, "pairs" of blocks, key "halves", or key "splits" (each in halves)."""
    group = c.head_count // c.head_count_kv
    kg = hfp.kernel_group(c.head_size, group)
    window = 0 if hfp.is_global_layer(c.architecture, layer) else c.sliding_window
    line = f"need {c.head_count_kv} {group // kg} {kg} {c.head_size} {window} {pos0} {n}\n"
    out = subprocess.run([_driver()], input=line, capture_output=True, text=True, check=True).stdout
    _, _, _, ksplit, _, _, groups, pairs, _ = map(int, out.split())
    if ksplit == 0:
        return ""
    return "splits" if ksplit > 1 else "one" if groups == 1 else "pairs" if pairs else "halves"
