"""Branching tables of so many regions that their configurations are more than
the work-items of one launch, against the same regions alone."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _regions(tb, count, size):
    g = tb.random_regular_graph(60, 3, seed=24)
    return tb.MISProblem(g), [tb.neighbor_region(g, [7 * i], size) for i in range(count)]


def test_tables(tb, backend):
    """258 regions of 24 vertices: 2^32 + 2^25 configurations."""
    p, regions = _regions(tb, 3, 24)
    alone = tb.branching_tables([(p, r) for r in regions], np.float32, backend=backend)
    many = tb.branching_tables([(p, r) for r in regions * 86], np.float32, backend=backend)
    assert len(many) == 258
    for i, t in enumerate(many):
        assert np.array_equal(t.alpha, alone[i % 3].alpha), i
        assert t.table == alone[i % 3].table, i
    assert all(len(t.table) > 1 for t in alone)


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
def test_alpha(tb, backend, dtype):
    """4098 regions of 24 vertices: 2^24 + 2^13 workgroups of their
    configurations."""
    from tensorbranching_jl_amd import _lib, branching
    p, regions = _regions(tb, 3, 24)
    n = 3 * 1366
    arr, keep, sizes = (_lib.TbhRegion * n)(), [], []
    for i, vs in enumerate(regions):
        vs, adj, ov, opos, _ = branching._region(p, vs, dtype)
        keep.append(np.ascontiguousarray(adj, np.uint32))
        sizes.append(1 << len(opos))
        for k in range(i, n, 3):
            arr[k].nv, arr[k].adj = len(vs), keep[-1].ctypes.data
            arr[k].open = sum(1 << o for o in opos)
    code = 0 if dtype == np.float32 else 1
    alone = np.empty(sum(sizes), dtype)
    many = np.empty(sum(sizes) * (n // 3), dtype)
    _lib.check(_lib.tbh().tbh_region_alpha(backend.handle, code, arr, 3, alone.ctypes.data))
    _lib.check(_lib.tbh().tbh_region_alpha(backend.handle, code, arr, n, many.ctypes.data))
    assert np.array_equal(many.reshape(-1, len(alone)), np.tile(alone, (n // 3, 1)))
    assert alone.max() > 0
