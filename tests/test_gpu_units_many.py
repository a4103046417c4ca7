"""A batch of more units than the workgroups of one launch."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def contract_edges(be, n):
    """n slices of one edge with weights 3 and 5, r = i mod 1009, each a unit."""
    from tensorbranching_jl_amd import _lib
    ix_ptr = np.array([0, 1, 2, 4], np.int32)
    ix = np.array([0, 1, 0, 1], np.int32)
    tree = np.array([0, 2, 3, 1], np.int32)
    weights = np.array([3, 5], np.float32)
    slices = (_lib.TbhSlice * n)()
    first = slices[0]
    first.nv, first.nleaves = 2, 3
    first.weights, first.ix_ptr = weights.ctypes.data, ix_ptr.ctypes.data
    first.ix, first.tree = ix.ctypes.data, tree.ctypes.data
    size = C.sizeof(_lib.TbhSlice)
    raw = np.frombuffer(slices, np.uint8).reshape(n, size)
    raw[1:] = raw[0]
    r = np.arange(n) % 1009
    raw[:, _lib.TbhSlice.r.offset:][:, :8] = r.astype(np.float64).view(np.uint8).reshape(n, 8)
    out = np.empty(n, np.float32)
    _lib.check(_lib.tbh().tbh_contract_slices(be.handle, 0, slices, n, out.ctypes.data, 1))
    return out, 5 + r.astype(np.float32)


def test_more_units_than_a_launch_holds(tb):
    """2^23 units of 512 work-items are 2^32 of them; a pool whose first batch
    takes every slice."""
    n = (1 << 23) + 3
    if os.sysconf("SC_AVPHYS_PAGES") * os.sysconf("SC_PAGE_SIZE") < 40 << 30:
        pytest.skip("needs 29 GB of host memory")
    with tb.HIPBackend(0, pool_bytes=64 << 30) as be:
        out, want = contract_edges(be, n)
        assert np.array_equal(out, want)
