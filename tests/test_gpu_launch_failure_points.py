"""Where a forced launch failure (TBH_INJECT_LAUNCH_FAILURE=N: the launch that
holds the wave of steps after N reports a failure) is found: at the first
launch, and at the very last one, which the end of a run waits for.  N counts
waves, more than there are launches, so the last launch is found by bisection.
A call of several batches, whose launches a thread issues, and one of a single
batch, which the caller issues itself; then a served round."""
import numpy as np
import pytest

from test_gpu_launch_failure import POOL, _backend, _slices

pytestmark = pytest.mark.gpu


def _fails(tb, br, at, pool):
    """Whether a contraction with the failure at `at` reports it, and its
    values, or those of the context's next contraction where it does."""
    import test_gpu_launch_failure as first
    old, first.POOL = first.POOL, pool
    try:
        be = _backend(tb, at)
    finally:
        first.POOL = old
    try:
        try:
            return False, be.contract_slices(br, np.float32, "batched")
        except tb.TbhError as ex:
            assert ex.code == -3 and "launch" in str(ex), (at, str(ex))
        return True, be.contract_slices(br, np.float32, "batched")
    finally:
        be.close()


@pytest.mark.parametrize("batches", ["several", "one"])
def test_first_and_last_launch(tb, orc, batches):
    br = _slices(tb)
    pool = POOL
    if batches == "one":
        br, pool = br[:3], 1 << 30
    ref = orc.contract_slices(br, np.float32)
    failed, got = _fails(tb, br, 0, pool)
    assert failed and np.array_equal(got, ref)
    lo, hi = 0, 1  # fails at lo; the first N that passes, by doubling
    while _fails(tb, br, hi, pool)[0]:
        lo, hi = hi, 2 * hi
        assert hi < 1 << 16
    while hi - lo > 1:
        mid = (lo + hi) // 2
        if _fails(tb, br, mid, pool)[0]:
            lo = mid
        else:
            hi = mid
    assert lo > 0
    # the last launch of the last batch, twice; past it nothing fails
    for _ in range(2):
        failed, got = _fails(tb, br, lo, pool)
        assert failed and np.array_equal(got, ref)
    failed, got = _fails(tb, br, hi, pool)
    assert not failed and np.array_equal(got, ref)


@pytest.mark.parametrize("at", [0, 1, 2])
def test_first_launches_of_a_served_round(tb, orc, at):
    br = _slices(tb)[:6]
    want = orc.contract_slices(br, np.float32).max()
    be = _backend(tb, at)
    try:
        with tb.Server(be) as srv:
            assert srv.wait(srv.submit(br)) == want
            st = srv.stats()
            assert st["retried_rounds"] >= 1 and st["failed_requests"] == 0, st
    finally:
        be.close()
