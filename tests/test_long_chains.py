"""Planning time of batched plans (csrc/tbh_plan.cpp) on long chains, whose
upper nodes hold more than a unit: linear in the chain's length (0.1 s for
10^5 leaves), where trying a unit at every node took half a minute."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_long_chains_plan_in_linear_time(tmp_path):
    gxx = shutil.which("g++")
    rocm_inc = "/opt/rocm/include"
    if gxx is None or not os.path.isdir(rocm_inc):
        pytest.skip("g++ or HIP headers not available")
    exe = tmp_path / "long_chain_check"
    csrc = os.path.join(ROOT, "tensorbranching.jl_amd", "csrc")
    cmd = [gxx, "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", os.path.join(ROOT, "include"),
           "-I", csrc, "-I", rocm_inc, os.path.join(ROOT, "tests", "host", "long_chain_check.cpp"),
           os.path.join(csrc, "tbh_plan.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe), "5"], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])
    assert [l.split()[0] for l in r.stdout.splitlines()] == ["chain", "bush", "halves"]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4000, 5000])
def test_chain_on_gpu(tb, backend, n):
    """A path's tree one vertex after another, as one unit and past it: the
    maximum independent set of a path of n vertices."""
    g = tb.SimpleGraph(n, [(v, v + 1) for v in range(n - 1)])
    nl = 2 * n - 1
    ix = list(range(n)) + [x for v in range(n - 1) for x in (v, v + 1)]
    ptr = list(range(n + 1)) + [n + 2 * (v + 1) for v in range(n - 1)]
    tree, x = [], 0
    for v in range(1, n):
        tree += [x, n + v - 1]
        x = nl + len(tree) // 2 - 1
        tree += [x, v]
        x = nl + len(tree) // 2 - 1
    code = tb.CompressedEinsum.from_arrays(np.asarray(ptr, np.int32), np.asarray(ix, np.int32),
                                           np.asarray(tree, np.int32))
    br = tb.SlicedBranch(tb.MISProblem(g), code, 0)
    for dtype in (np.float32, np.int32):
        assert backend.contract_slices([br], dtype)[0] == (n + 1) // 2
