"""The size rules that pick the N-D executor's kernels, on the CPU (tests/cpp/test_nd_rules.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "wgpu-ocr_amd", "csrc")
ROCM_INC = "/opt/rocm/include"


def test_nd_rules(tmp_path):
    if shutil.which("g++") is None or not os.path.isdir(ROCM_INC):
        pytest.skip("g++ or the HIP headers are not available")
    exe = str(tmp_path / "nd_rules")
    cmd = ["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", CSRC, "-I", ROCM_INC,
           os.path.join(ROOT, "tests", "cpp", "test_nd_rules.cpp"), "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stdout
