"""Slices whose default plan does not fit the pool run by their lean plan
(PlanOptions::lean): batched calls, served requests and plain calls on pools
between the two arenas, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _slices(tb, n, sc, seed, pick):
    g = tb.random_regular_graph(n, 3, seed=seed)
    br = tb.slice_graph(g, None, tb.ContractionTreeSlicer(sc_target=sc, order_trials=10),
                        seed=seed)
    return [[b for b in br if b.code is not None][i] for i in pick]


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
def test_batched(tb, orc, dtype):
    """Arenas of 14.3 and 18.5 MB; a batch's region of 17.25 MB."""
    br = _slices(tb, 160, 21, 1, (1, 0, 1, 2))
    assert tb.slice_footprint(br[0], dtype) > (69 << 20) // 4
    ref = orc.contract_slices(br, dtype)
    with tb.HIPBackend(0, pool_bytes=23 << 20) as be:
        assert np.array_equal(be.contract_slices(br, dtype, "batched"), ref)
        assert np.array_equal(be.contract_slices(br[:1], dtype, "batched"), ref[:1])


def test_served(tb, orc):
    br = _slices(tb, 160, 21, 1, (1, 0, 2))
    want = orc.contract_slices(br, np.float32).max()
    with tb.HIPBackend(0, pool_bytes=23 << 20) as be:
        with tb.Server(be) as srv:
            t = srv.submit(br)
            assert srv.wait(t) == want
            assert srv.stats()["failed_requests"] == 0


def test_plain(tb, orc):
    """Arenas of 31.4 and 32.5 MB, 0.9 MB of descriptors; a pool of 32.4 MB."""
    br = _slices(tb, 200, 21, 4, (5,))
    ref = orc.contract_slices(br, np.float32)
    with tb.HIPBackend(0, pool_bytes=32400000) as be:
        assert np.array_equal(be.contract_slices(br, np.float32, "plain"), ref)


def test_too_large_is_refused(tb):
    """A pool that holds neither plan refuses the slice, as before."""
    br = _slices(tb, 160, 21, 1, (1,))
    with tb.HIPBackend(0, pool_bytes=16 << 20) as be:
        for mode in ("batched", "plain"):
            with pytest.raises(tb.TbhError) as ex:
                be.contract_slices(br, np.float32, mode)
            assert ex.value.code == -2, mode
