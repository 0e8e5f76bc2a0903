"""The compiled passes' four-step twiddles are off by their two factors' single
roundings only (tests/host/twiddle_check.cpp, compiled with the host compiler)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include/hip"),
                    reason="needs g++ and the HIP headers")
def test_twiddle_progression(tmp_path):
    exe = str(tmp_path / "twiddle_check")
    cmd = ["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unknown-pragmas", "-D__HIP_PLATFORM_AMD__", "-I",
           os.path.join(ROOT, "radis_amd", "csrc"), "-I", "/opt/rocm/include",
           os.path.join(ROOT, "tests", "host", "twiddle_check.cpp"), "-o", exe]
    p = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stderr[-3000:]
    p = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, (p.stdout, p.stderr)
