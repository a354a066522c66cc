"""plan_stack (csrc/rt_common.hpp): what part of a traversal stack is in LDS,
for every depth and every setting.  A launch that spills sizes its area by
need - lds entries and a launch that does not must hold them all, so either
mistake is an access out of bounds."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "vulkan-compute-ray-tracing_amd", "csrc")


def test_every_stack_has_room(tmp_path):
    gxx, rocm_inc = shutil.which("g++"), "/opt/rocm/include"
    if gxx is None or not os.path.isdir(rocm_inc):
        pytest.skip("g++ or the ROCm headers are not present")
    out = str(tmp_path / "stack_plan")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", rocm_inc, "-I",
                        os.path.join(ROOT, "include"), "-I", CSRC,
                        os.path.join(ROOT, "tests", "cpp", "stack_plan_check.cpp"), "-o", out],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    rows = [tuple(map(int, line.split())) for line in subprocess.run([out], capture_output=True, text=True,
                                                                     check=True).stdout.splitlines()]
    assert len(rows) == 96 * 4 * 2
    for need, asked, crowded, lds, deep in rows:
        if deep:
            assert lds in (8, 16, 24, 32) and need > lds
        else:
            assert lds in (24, 36, 48, 64, 96) and need <= lds
        if asked:
            # as many in LDS as asked for, or all of them
            assert (deep and lds == asked) if asked < need else not deep
        else:
            assert bool(deep) == (bool(crowded) and need > 24)
