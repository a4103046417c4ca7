"""The planner's plans of less memory (PlanOptions::lean): their arenas are
those of the plan of one step per tree node and wave, whatever the default
plan gains its speed by."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# (n, sc, seed): lean arena bytes of the first six slices, batched and plain
ARENAS = {
    (160, 21, 1): ([13750784, 14333952, 11055616, 12587264, 7488512, 18002176],
                   [18761216, 34087424, 16785408, 33758464, 9970688, 29369088]),
    (200, 21, 4): ([23225600, 27320832, 29562112, 27959552, 27280896, 25141504],
                   [41955328, 37498624, 41708288, 35399424, 35667968, 31434240]),
}


def _write_slices(path, branches):
    with open(path, "wb") as f:
        f.write(np.int32(len(branches)).tobytes())
        for b in branches:
            c = b.code
            tree = np.asarray(c.tree, np.int32)
            f.write(np.asarray([b.p.g.nv, c.nleaves, len(c.ix_ptr), len(c.ix), len(tree)],
                               np.int32).tobytes())
            for a in (c.ix_ptr, c.ix, tree):
                f.write(np.ascontiguousarray(a, np.int32).tobytes())


@pytest.mark.parametrize("key", sorted(ARENAS))
def test_lean_arenas(tb, tmp_path, key):
    gxx = shutil.which("g++")
    rocm_inc = "/opt/rocm/include"
    if gxx is None or not os.path.isdir(rocm_inc):
        pytest.skip("g++ or HIP headers not available")
    exe = tmp_path / "lean_check"
    csrc = os.path.join(ROOT, "tensorbranching.jl_amd", "csrc")
    cmd = [gxx, "-O1", "-g", "-std=c++17", "-fsanitize=address,undefined",
           "-fno-sanitize-recover=all", "-D__HIP_PLATFORM_AMD__", "-I",
           os.path.join(ROOT, "include"), "-I", csrc, "-I", rocm_inc,
           os.path.join(ROOT, "tests", "host", "lean_check.cpp"),
           os.path.join(csrc, "tbh_plan.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    n, sc, seed = key
    g = tb.random_regular_graph(n, 3, seed=seed)
    br = tb.slice_graph(g, None, tb.ContractionTreeSlicer(sc_target=sc, order_trials=10),
                        seed=seed)
    br = [b for b in br if b.code is not None][:6]
    _write_slices(str(tmp_path / "slices.bin"), br)
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")
    r = subprocess.run([str(exe), str(tmp_path / "slices.bin")], capture_output=True, text=True,
                       env=env, timeout=600)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])
    rows = [tuple(map(int, l.split())) for l in r.stdout.splitlines()]
    assert [x[1] for x in rows[0::2]] == ARENAS[key][0]
    assert [x[1] for x in rows[1::2]] == ARENAS[key][1]
    # the default plan of some of them needs more
    assert any(x[0] > x[1] for x in rows)
