"""Subtrees contracted in LDS by one workgroup (csrc/tbh_unit.hip) against
the oracle, bit for bit.  Random pairings of a graph's leaves give trees whose
nodes reach and pass every limit of a unit: 15 union labels, 14 output labels,
6 reduced labels, 2^17 MACs and 8192 LDS elements, so that slices come out as
one unit, as many units below and above larger steps (which then read tensors from
memory), and as leaves read by those steps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _random_code(tb, g, rng, local):
    """All leaves paired at random; `local` prefers pairs near each other,
    which keeps more of the tree small."""
    ixs = [[v] for v in range(g.nv)] + [[int(u), int(v)] for u, v in g.edges]
    nodes = [(min(x), i) for i, x in enumerate(ixs)]
    while len(nodes) > 1:
        if local:
            nodes.sort(key=lambda t: t[0])
            i = int(rng.integers(len(nodes) - 1))
            j = i + 1
        else:
            i, j = sorted(int(k) for k in rng.choice(len(nodes), 2, replace=False))
        b = nodes.pop(j)
        a = nodes.pop(i)
        nodes.append((min(a[0], b[0]), tb.ContractionTree(a[1], b[1])))
    return tb.CompressedEinsum(ixs, [], nodes[0][1])


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("nv,degree,local", [(1, 0, False), (2, 1, False), (5, 2, True),
                                             (9, 3, False), (13, 4, False), (14, 3, False),
                                             (15, 4, False), (16, 3, True), (17, 4, False),
                                             (19, 3, False), (40, 3, True)])
def test_random_trees(tb, orc, backend, nv, degree, local, dtype):
    rng = np.random.default_rng(1000 * nv + 10 * degree + local)
    branches = []
    for _ in range(8):
        ne = min(nv * degree // 2, nv * (nv - 1) // 2)
        pairs = [(u, v) for u in range(nv) for v in range(u + 1, nv)]
        pick = rng.choice(len(pairs), ne, replace=False) if ne else []
        g = tb.SimpleGraph(nv, [pairs[int(k)] for k in pick])
        w = rng.integers(1, 101, nv).astype(dtype)
        branches.append(tb.SlicedBranch(tb.MISProblem(g, w), _random_code(tb, g, rng, local),
                                        int(rng.integers(0, 9))))
    if nv in (17, 19):
        # units above larger steps: unit steps (no tile) past the first wave
        steps = [st for b in branches for st in tb.plan_steps(b, dtype)]
        assert any(st["kind"] == 0 and st["level"] > 1 and st["rank_c"] > 0 and
                   st["tile_bits"] == 0 for st in steps)
        assert any(st["tile_bits"] > 0 for st in steps)
    print(f"[units] nv={nv} sc={[int(tb.sc(b)) for b in branches if len(b.code.tree)]}",
          flush=True)
    assert np.array_equal(backend.contract_slices(branches, dtype),
                          orc.contract_slices(branches, dtype))


@pytest.mark.parametrize("leaves", [5, 7, 8, 9])
def test_star_reduced_at_once(tb, orc, backend, leaves):
    """The two halves of K_{n,n} meet in one step that reduces n labels held
    by both: up to a unit's 6, then past them."""
    n = leaves
    g = tb.SimpleGraph(2 * n, [[i, n + j] for i in range(n) for j in range(n)])
    ixs = [[v] for v in range(2 * n)] + [[int(u), int(v)] for u, v in g.edges]
    edge = {tuple(map(int, e)): 2 * n + k for k, e in enumerate(g.edges)}

    def chain(items):
        t = items[0]
        for x in items[1:]:
            t = tb.ContractionTree(t, x)
        return t

    left = chain([edge[i, n + j] for i in range(n) for j in range(n // 2)] + list(range(n)))
    right = chain([edge[i, n + j] for i in range(n) for j in range(n // 2, n)] +
                  list(range(n, 2 * n)))
    code = tb.CompressedEinsum(ixs, [], tb.ContractionTree(left, right))
    w = np.random.default_rng(n).integers(1, 101, 2 * n)
    for dtype in (np.float32, np.int32):
        b = tb.SlicedBranch(tb.MISProblem(g, w.astype(dtype)), code, 3)
        assert np.array_equal(backend.contract_slices([b], dtype), orc.contract_slices([b], dtype))


@pytest.mark.parametrize("nv", [32, 33, 34, 64, 66, 200])
def test_long_chain(tb, orc, backend, nv):
    """A path contracted from one end: a unit of 2 nv - 2 levels of one step
    each, all of one wave's, which reads its shares 64 at a time."""
    g = tb.SimpleGraph(nv, [(i, i + 1) for i in range(nv - 1)])
    ixs = [[v] for v in range(nv)] + [[int(u), int(v)] for u, v in g.edges]
    t = 0
    for i in range(nv - 1):
        t = tb.ContractionTree(tb.ContractionTree(t, nv + i), i + 1)
    code = tb.CompressedEinsum(ixs, [], t)
    w = np.random.default_rng(nv).integers(1, 101, nv)
    for dtype in (np.float32, np.int32):
        b = tb.SlicedBranch(tb.MISProblem(g, w.astype(dtype)), code, 3)
        assert np.array_equal(backend.contract_slices([b], dtype), orc.contract_slices([b], dtype))


def test_infinite_weights(tb, backend):
    """A vertex of weight -inf is never taken; one of +inf is."""
    g = tb.random_regular_graph(20, 3, seed=4)
    code = tb.initialize_code(g, 10)
    w = np.ones(20, np.float32)
    w[3] = -np.inf
    v = np.ones(20, np.float32)
    v[3] = -100
    pair = [tb.SlicedBranch(tb.MISProblem(g, x), code, 0) for x in (w, v)]
    got = backend.contract_slices(pair)
    assert got[0] == got[1]
    w[3] = np.inf
    assert backend.solve_slice(tb.SlicedBranch(tb.MISProblem(g, w), code, 0)) == np.inf
