"""GEMM steps beside a level's other steps on a second stream, where both are
long, or behind them (csrc/tbh_runtime.cpp): batches whose levels are all
short, of both kinds, and mostly long, repeated, against the same batch on one
stream and a slice of it against the oracle, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 12, 100, 400])
def test_levels_on_two_streams(tb, orc, backend, count):
    g = tb.random_regular_graph(200, 3, seed=1)
    br = tb.slice_graph(g, None, tb.ContractionTreeSlicer(sc_target=20, order_trials=10), seed=1)
    br = sorted((b for b in br if b.code is not None), key=lambda b: -tb.complexity(b).tc)
    steps = tb.plan_steps(br[0], np.int32)
    assert {s["kind"] for s in steps} >= {0, 1}
    rng = np.random.default_rng(count)
    pick = [tb.SlicedBranch(tb.MISProblem(b.p.g, rng.integers(1, 101, b.p.g.nv).astype(np.int32)),
                            b.code, b.r) for b in (br * (count // len(br) + 1))[:count]]
    t0 = backend.tuning()
    try:
        backend.set_tuning(**dict(t0, concurrent=0))
        want = backend.contract_slices(pick, np.int32)
    finally:
        backend.set_tuning(**t0)
    for _ in range(3):
        assert np.array_equal(backend.contract_slices(pick, np.int32), want)
    assert want[0] == orc.contract_slices(pick[:1], np.int32)[0]
