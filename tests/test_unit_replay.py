"""The LDS plans of units replayed on the host (tests/host/unit_replay.cpp):
sliced networks of several graph families, and random trees over random
graphs, whose units are shaped otherwise."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _random_tree(rng, nv, ne, local):
    """A random MIS network and contraction tree: (nv, ix_ptr, ix, tree)."""
    edges = set()
    while len(edges) < ne:
        u, v = (int(x) for x in rng.integers(0, nv, 2))
        if u != v:
            edges.add((min(u, v), max(u, v)))
    leaves = [[v] for v in range(nv)] + [list(e) for e in sorted(edges)]
    ptr = np.cumsum([0] + [len(x) for x in leaves])
    # joins of neighbours in an order by label (local) or of any two
    alive = sorted(range(len(leaves)), key=lambda i: leaves[i]) if local else \
        list(range(len(leaves)))
    tree, nxt = [], len(leaves)
    while len(alive) > 1:
        if local:
            k = int(rng.integers(0, len(alive) - 1))
            a, b = alive[k], alive.pop(k + 1)
        else:
            k = int(rng.integers(0, len(alive)))
            a = alive.pop(k)
            k = int(rng.integers(0, len(alive)))
            b = alive[k]
        alive[k] = nxt
        tree += [a, b]
        nxt += 1
    return nv, ptr, [x for l in leaves for x in l], tree


def test_units_replayed(tb, tmp_path):
    gxx = shutil.which("g++")
    rocm_inc = "/opt/rocm/include"
    if gxx is None or not os.path.isdir(rocm_inc):
        pytest.skip("g++ or HIP headers not available")
    exe = tmp_path / "unit_replay"
    csrc = os.path.join(ROOT, "tensorbranching.jl_amd", "csrc")
    cmd = [gxx, "-O2", "-g", "-std=c++17", "-fsanitize=address,undefined",
           "-fno-sanitize-recover=all", "-D__HIP_PLATFORM_AMD__", "-I",
           os.path.join(ROOT, "include"), "-I", csrc, "-I", rocm_inc,
           os.path.join(ROOT, "tests", "host", "unit_replay.cpp"),
           os.path.join(csrc, "tbh_plan.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    items = []
    graphs = [(tb.random_regular_graph(100, 3, seed=0), 10),
              (tb.random_regular_graph(160, 3, seed=5), 18), (tb.random_ksg(14, 14, 0.8, seed=1), 14),
              (tb.erdos_renyi(40, 0.12, seed=2), 12)]
    for g, sc in graphs:
        br = tb.slice_graph(g, None, tb.ContractionTreeSlicer(sc_target=sc, order_trials=5), seed=1)
        items += [(b.p.g.nv, b.code.ix_ptr, b.code.ix, b.code.tree)
                  for b in br[:8] if b.code is not None]
    rng = np.random.default_rng(7)
    for k in range(150):
        nv = int(rng.integers(2, 60))
        ne = int(rng.integers(1, 1 + min(2 * nv, nv * (nv - 1) // 2)))
        items.append(_random_tree(rng, nv, ne, k % 3 != 0 or nv > 16))
    path = tmp_path / "slices.bin"
    with open(path, "wb") as f:
        f.write(np.int32(len(items)).tobytes())
        for nv, ptr, ix, tree in items:
            f.write(np.asarray([nv, len(ptr) - 1, len(ptr), len(ix), len(tree)],
                               np.int32).tobytes())
            for a in (ptr, ix, tree):
                f.write(np.ascontiguousarray(a, np.int32).tobytes())
    env = dict(os.environ, ASAN_OPTIONS="verify_asan_link_order=0")
    r = subprocess.run([str(exe), str(path)], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-4000:])
    plans, units, mixed, moved, noticed = (int(x) for x in r.stdout.split()[::2])
    # (a unit of two levels without a dependency can be moved unnoticed)
    assert plans > 120 and units > 200 and mixed > 20 and noticed > 0.9 * moved > 100
