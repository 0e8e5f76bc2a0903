"""The half-length rule, its workspace and its work items (ldm_plan.h),
compiled with the host compiler and swept on the CPU."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"),
                    reason="needs g++ and the HIP headers")
def test_half_length_plans(tmp_path):
    exe = str(tmp_path / "half_check")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unused-function", "-D__HIP_PLATFORM_AMD__", "-I",
           os.path.join(ROOT, "radis_amd", "csrc"), "-I", os.path.join(ROOT, "include"), "-I", "/opt/rocm/include",
           os.path.join(ROOT, "tests", "host", "half_check.cpp"), "-o", exe, "-lpthread"]
    p = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-3000:]
    p = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(p.stdout)
    assert p.returncode == 0, p.stderr[-3000:] + p.stdout
