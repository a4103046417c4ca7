"""The standalone GEMM's dispatch (csrc/tbh_gemm_rule.hpp) checked on the host:
which products run in which tiles, and that their K ranges cover K."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_gemm_rule(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    rocm_inc = "/opt/rocm/include"
    if not os.path.isdir(rocm_inc):
        pytest.skip("HIP headers not available")
    exe = tmp_path / "gemm_rule_check"
    cmd = [gxx, "-O1", "-g", "-std=c++17", "-fsanitize=undefined", "-fno-sanitize-recover=all",
           "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "tensorbranching.jl_amd", "csrc"),
           "-I", rocm_inc, os.path.join(ROOT, "tests", "host", "gemm_rule_check.cpp"),
           "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])
    assert "checked" in r.stdout
