"""plan_launch (csrc/rt_common.hpp) around its boundaries: the grid is never
exceeded, waves that get their rays at the start have a lane for each, and a
kernel that plans again from its own grid finds the host's plan."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "vulkan-compute-ray-tracing_amd", "csrc")


def test_launch_plans(tmp_path):
    gxx, rocm_inc = shutil.which("g++"), "/opt/rocm/include"
    if gxx is None or not os.path.isdir(rocm_inc):
        pytest.skip("g++ or the ROCm headers are not present")
    out = str(tmp_path / "launch_plan")
    r = subprocess.run([gxx, "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", rocm_inc, "-I",
                        os.path.join(ROOT, "include"), "-I", CSRC,
                        os.path.join(ROOT, "tests", "cpp", "launch_plan_check.cpp"), "-o", out],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    lines = subprocess.run([out], capture_output=True, text=True, check=True).stdout.splitlines()
    assert len(lines) == 1 and int(lines[0]) > 1000, lines[:5]
