"""tbh_region_alpha against the contraction it stands for (one slice per
boundary configuration through the batched contraction) and the brute-force
tables: no open vertex, all of them open, more boundary bits than the
kernel's LDS table holds, one workgroup of configurations and several,
negative weights, an empty region, and the Int32 bound."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _alpha(tb, backend, g, vs, w, dtype):
    from tensorbranching_jl_amd import _lib, branching
    vs, adj, ov, opos, ww = branching._region(tb.MISProblem(g, w), vs, np.dtype(dtype).type)
    reg = (_lib.TbhRegion * 1)()
    reg[0].nv, reg[0].open = len(vs), sum(1 << k for k in opos)
    a, ww = np.ascontiguousarray(adj), np.ascontiguousarray(ww)
    reg[0].adj = a.ctypes.data if len(vs) else None
    reg[0].weights = ww.ctypes.data if w is not None else None
    out = np.empty(1 << len(opos), dtype)
    code = 0 if dtype == np.float32 else 1
    _lib.check(_lib.tbh().tbh_region_alpha(backend.handle, code, reg, 1, out.ctypes.data))
    return vs, adj, opos, ww, out


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("n,size,degree", [(12, 12, 3), (14, 1, 3), (40, 11, 3), (60, 12, 3),
                                           (60, 13, 3), (400, 13, 12), (80, 17, 3)])
def test_equals_the_contraction(tb, backend, n, size, degree, dtype):
    rng = np.random.default_rng(n + size)
    g = tb.erdos_renyi(n, degree / n, seed=n) if degree > 3 else \
        tb.random_regular_graph(n, degree, seed=n + size)
    vs = list(range(n)) if size == n else \
        [int(v) for v in rng.choice(n, size, replace=False)] if degree > 3 else \
        tb.neighbor_region(g, [0], size)
    for w in (None, rng.integers(-20, 60, n).astype(dtype)):
        vs, adj, opos, ww, got = _alpha(tb, backend, g, vs, w, dtype)
        zero = -np.inf if dtype == np.float32 else tb.TBH_I32_NEG_INF
        want = np.full(len(got), zero, dtype)
        slices, where = [], []
        for b in range(len(got)):
            chosen = [opos[k] for k in range(len(opos)) if (b >> k) & 1]
            if any(int(adj[c]) >> d & 1 for c in chosen for d in chosen):
                continue
            gone = set(opos) | {v for c in chosen for v in range(len(vs)) if int(adj[c]) >> v & 1}
            keep = [v for v in range(len(vs)) if v not in gone]
            sub = tb.SimpleGraph(len(keep), [(i, j) for j, v in enumerate(keep)
                                             for i, u in enumerate(keep[:j]) if int(adj[u]) >> v & 1])
            code = tb.initialize_code(sub, 1) if keep else None
            slices.append(tb.SlicedBranch(tb.MISProblem(sub, ww[keep] if keep else None), code,
                                          int(sum(ww[c] for c in chosen))))
            where.append(b)
        want[where] = backend.contract_slices(slices, dtype)
        assert np.array_equal(got, want)


def test_wide_boundary_against_bruteforce(tb, orc, backend):
    g = tb.erdos_renyi(400, 12 / 400, seed=8)
    vs = [int(v) for v in np.random.default_rng(8).choice(400, 14, replace=False)]
    for dtype in (np.float32, np.int32):
        t = tb.branching_table(tb.MISProblem(g), vs, dtype, backend=backend)
        assert len(t.open_vertices) == 14
        ov, _, red, rows = orc.branching_table_bruteforce(g, None, vs)
        got = np.asarray(t.alpha, np.float64)
        got[got <= tb.TBH_I32_NEG_INF] = -np.inf
        assert t.open_vertices == ov and got.tolist() == red.tolist() and t.table == rows


def test_empty_region_and_int32_bound(tb, backend):
    g = tb.random_regular_graph(24, 3, seed=2)
    t = tb.branching_table(tb.MISProblem(g), [], backend=backend)
    assert t.alpha.tolist() == [0.0] and t.table == [[0]]
    w = np.full(24, (1 << 24) - 1, np.int32)  # 24 of them pass 2^28
    with pytest.raises(tb.TbhError, match="2\\^28"):
        tb.branching_table(tb.MISProblem(g, w), list(range(24)), np.int32, backend=backend)
    t = tb.branching_table(tb.MISProblem(g, w), list(range(15)), np.int32, backend=backend)
    assert max(t.alpha) < 1 << 28
