"""GEMM steps in 64 x 64 tiles (csrc/tbh_gemm.hip, the steps of a batched plan
with few tiles): slices whose plans hold such steps at K = 16 (half a slab),
32 (one slab), 64 and more, storing column-major, as row quads and through
LDS, against the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
def test_small_gemm_steps(tb, orc, backend, dtype):
    g = tb.random_regular_graph(200, 3, seed=1)
    br = tb.slice_graph(g, None, tb.ContractionTreeSlicer(sc_target=18, order_trials=10), seed=1)
    rng = np.random.default_rng(3)
    seen, pick = set(), []
    for b in sorted((b for b in br if b.code is not None), key=lambda b: tb.complexity(b).tc):
        kinds = {(s["gemm_store"], min(s["K"], 128)) for s in tb.plan_steps(b, dtype)
                 if s["kind"] == 1 and min(s["M"], s["N"]) >= 64 and
                 s["M"] * s["N"] * s["batch"] < 256 << 12}
        if kinds - seen:
            seen |= kinds
            w = rng.integers(1, 101, b.p.g.nv).astype(dtype)
            pick.append(tb.SlicedBranch(tb.MISProblem(b.p.g, w), b.code, b.r))
    assert {s for s, _ in seen} == {0, 1, 2} and {k for _, k in seen} == {16, 32, 64, 128}
    assert np.array_equal(backend.contract_slices(pick, dtype), orc.contract_slices(pick, dtype))
