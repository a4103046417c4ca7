"""Branching tables of regions: the table step of optimal_branches
(src/branch.jl:79, branching_table(p, TensorNetworkSolver(), region) from
OptimalBranchingMIS), batched over many regions.

For a region (a vertex list of a MIS problem) the boundary ("open")
vertices are those with a neighbour outside it.  Its alpha tensor holds, per
boundary configuration b (bit k = the k-th open vertex in region order),
the best weight of an independent set of the region whose boundary part is
b: the SizeMax contraction of the region's tensor network with its open
labels kept.  tbh_region_alpha computes it for every region in one
launch by enumerating the region's configurations (at most 2^24), which the
table's rows need anyway.  tbh_region_tables then prunes each tensor as
mis_compactify! does (an entry that a proper subset of its boundary
configuration matches or beats becomes the tropical zero) and enumerates, for
each surviving b, every region configuration that reaches it: the rows of the
table.  All of it runs on the GPU.

Exact parity with OptimalBranchingMIS (not vendored here) is unpinned; the
tests pin the tables against brute-force enumeration of every region
configuration and against hand-worked examples.
"""
import ctypes as C

import numpy as np

from . import _lib
from ._lib import check
from .api import _dtype_code, default_backend


def open_vertices(g, vs):
    """The vertices of vs with a neighbour outside vs, in vs order."""
    edges = np.asarray(g.edges).reshape(-1, 2)
    inside = np.isin(edges, [int(v) for v in vs])
    crossing = set(edges[inside & ~inside[:, ::-1]].tolist())
    return [int(v) for v in vs if int(v) in crossing]


def neighbor_region(g, seeds, n_max):
    """A region grown from `seeds` by breadth-first layers (lowest vertex id
    first within a layer) until it holds n_max vertices."""
    nb = [[] for _ in range(g.nv)]
    for u, v in np.asarray(g.edges).reshape(-1, 2):
        nb[int(u)].append(int(v))
        nb[int(v)].append(int(u))
    region = []
    seen = set()
    layer = sorted(set(int(s) for s in seeds))
    while layer and len(region) < n_max:
        nxt = set()
        for v in layer:
            if v in seen:
                continue
            if len(region) == n_max:
                break
            seen.add(v)
            region.append(v)
            nxt.update(nb[v])
        layer = sorted(nxt - seen)
    return region


class BranchingTable:
    """The table of one region: `vertices` (the region), `open_vertices`,
    `alpha` (the reduced alpha tensor, one value per boundary configuration,
    the tropical zero where pruned) and `table` (one row per surviving
    boundary configuration, ascending; a row lists the region
    configurations reaching it as bitmasks, bit i = vertices[i])."""

    def __init__(self, vertices, open_vertices, alpha, table):
        self.vertices = list(vertices)
        self.open_vertices = list(open_vertices)
        self.bit_length = len(self.vertices)
        self.alpha = alpha
        self.table = table

    def __repr__(self):
        return (f"BranchingTable(bit_length={self.bit_length}, open={len(self.open_vertices)}, "
                f"rows={len(self.table)})")


def _region(p, vs, npdt):
    vs = [int(v) for v in vs]
    pos = {v: i for i, v in enumerate(vs)}
    if len(pos) != len(vs):
        raise ValueError("a region lists a vertex twice")
    nv = len(vs)
    adj = np.zeros(max(1, nv), np.uint32)
    edges = np.asarray(p.g.edges).reshape(-1, 2)
    for u, v in edges[np.isin(edges, vs).all(axis=1)].tolist():
        adj[pos[u]] |= np.uint32(1 << pos[v])
        adj[pos[v]] |= np.uint32(1 << pos[u])
    ov = open_vertices(p.g, vs)
    opos = [pos[v] for v in ov]
    if p.weights is None:
        w = np.ones(nv, npdt)
    else:
        w = np.asarray(p.weights)[vs].astype(npdt)
    return vs, adj[:nv] if nv else adj[:0], ov, opos, w


def branching_tables(items, element_type=np.float32, backend=None, order_trials=4, seed=0):
    """Branching tables of many regions at once: items = [(MISProblem,
    region vertex list), ...] -> [BranchingTable, ...].  Every region's alpha
    tensor, its pruning and its rows come from the GPU (tbh_region_alpha,
    tbh_region_tables).  order_trials and seed, which tune a search for
    contraction trees, have no effect on the tables."""
    be = backend or default_backend()
    code, npdt = _dtype_code(element_type)
    regions = []
    for p, vs in items:
        vs, adj, ov, opos, w = _region(p, vs, npdt)
        if len(vs) > 24 or len(ov) > 16:
            raise ValueError("a region needs at most 24 vertices and 16 open vertices")
        regions.append((vs, adj, ov, opos, w))
    arr = (_lib.TbhRegion * max(1, len(regions)))()
    keep = []
    for i, (vs, adj, ov, opos, w) in enumerate(regions):
        a = np.ascontiguousarray(adj, np.uint32)
        keep.append(a)
        arr[i].nv = len(vs)
        arr[i].adj = a.ctypes.data if len(vs) else None
        if items[i][0].weights is not None:
            ww = np.ascontiguousarray(w, npdt)
            keep.append(ww)
            arr[i].weights = ww.ctypes.data
        else:
            arr[i].weights = None
        arr[i].open = sum(1 << k for k in opos)
    n = len(regions)
    a0 = np.cumsum([0] + [1 << len(R[3]) for R in regions])
    alpha = np.empty(max(1, int(a0[-1])), npdt)
    check(_lib.tbh().tbh_region_alpha(be.handle, code, arr, n, alpha.ctypes.data))
    # the rows, into a buffer most calls fit; else once more with their number
    gptr = np.zeros(n + 1, np.uint64)
    total = C.c_size_t()
    reduced = alpha.copy()
    cap = min(sum(1 << len(R[0]) for R in regions), 1 << 20)
    cfg = np.empty(max(1, cap), np.uint32)
    rc = _lib.tbh().tbh_region_tables(be.handle, code, arr, n, reduced.ctypes.data,
                                      gptr.ctypes.data, cfg.ctypes.data, cap, C.byref(total))
    if rc == _lib.TBH_ENOMEM and total.value > cap:
        cfg = np.empty(total.value, np.uint32)
        reduced = alpha.copy()
        rc = _lib.tbh().tbh_region_tables(be.handle, code, arr, n, reduced.ctypes.data,
                                          gptr.ctypes.data, cfg.ctypes.data, total.value,
                                          C.byref(total))
    check(rc)
    out = []
    for i, (vs, adj, ov, opos, w) in enumerate(regions):
        red = reduced[a0[i]:a0[i + 1]]
        x = cfg[int(gptr[i]):int(gptr[i + 1])]
        # ordered by boundary configuration, then ascending: a row each
        b = np.zeros(len(x), np.uint32)
        for k, at in enumerate(opos):
            b |= ((x >> np.uint32(at)) & np.uint32(1)) << np.uint32(k)
        rows = x.tolist()
        cuts = [0] + (np.flatnonzero(b[1:] != b[:-1]) + 1).tolist() + [len(rows)]
        table = [rows[s:e] for s, e in zip(cuts, cuts[1:]) if e > s]
        out.append(BranchingTable(vs, ov, red.copy(), table))
    return out


def branching_table(p, region, element_type=np.float32, backend=None, **kw):
    """branching_table(p, TensorNetworkSolver(), region) for one region."""
    return branching_tables([(p, region)], element_type, backend, **kw)[0]
