"""Timed cases of the framework's public entry points, small calls to the
largest: max-plus GEMMs, single slices, sliced MIS networks, a burst of
served requests and the branching tables of a graph's regions.

A network's graph, slices and contraction trees follow from the case alone;
the vertex weights and the slices' fixed weights r are drawn from the seed.
"""
import functools
import importlib.util
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
NAME = "tensorbranching_jl_amd"
I32_ZERO = -(1 << 30)  # the tropical zero of Int32
# device pools of the contraction backend and of the serving one
POOL, SERVE_POOL = 80 << 30, 16 << 30
# a drawn network holds at most this many slices and log2 MACs
MAX_SLICES, MAX_LOG2_MACS = 800, 39.0


def package():
    if NAME not in sys.modules:
        d = os.path.join(ROOT, "tensorbranching.jl_amd")
        spec = importlib.util.spec_from_file_location(
            NAME, os.path.join(d, "__init__.py"), submodule_search_locations=[d])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[NAME] = mod
        spec.loader.exec_module(mod)
    return sys.modules[NAME]


@functools.lru_cache(None)
def backend():
    return package().HIPBackend(0, pool_bytes=POOL)


@functools.lru_cache(None)
def server():
    return package().Server(package().HIPBackend(0, pool_bytes=SERVE_POOL))


# ------------------------------------------------------------- the cases ---
def listed():
    return [
        # the lower seam mul!(C, A, B): the latency of one small product
        {"name": "gemm_64", "kind": "gemm", "M": 64, "N": 64, "K": 64, "batch": 1,
         "dtype": "float32"},
        # an ordinary square product (too few 128 x 128 tiles to fill the chip)
        {"name": "gemm_512", "kind": "gemm", "M": 512, "N": 512, "K": 512, "batch": 1,
         "dtype": "float32"},
        # a ragged batched product, Int32 (no dimension a multiple of 4)
        {"name": "gemm_i32_ragged", "kind": "gemm", "M": 1021, "N": 515, "K": 777, "batch": 3,
         "dtype": "int32"},
        # the largest product of the GEMM configuration
        {"name": "gemm_4096", "kind": "gemm", "M": 4096, "N": 4096, "K": 4096, "batch": 1,
         "dtype": "float32"},
        # a caller blocked on one small slice (solve_slice in slice_dfs_lp)
        {"name": "solve_slice", "kind": "solve", "graph": "regular", "n": 100, "gseed": 0,
         "sc": 15, "trials": 20, "dtype": "float32", "weights": "int"},
        # the small benchmark configuration: 3-regular n=100 sliced to sc 10
        {"name": "slices_n100_sc10", "kind": "contract", "graph": "regular", "n": 100,
         "gseed": 0, "sc": 10, "trials": 20, "dtype": "float32", "weights": "unit"},
        # many medium slices, Int32 weights
        {"name": "slices_n200_sc20_i32", "kind": "contract", "graph": "regular", "n": 200,
         "gseed": 1, "sc": 20, "trials": 10, "dtype": "int32", "weights": "int"},
        # one unsliced network: 3-regular n=200, contracted whole
        {"name": "whole_n200", "kind": "contract", "graph": "regular", "n": 200, "gseed": 1,
         "sc": 29, "trials": 100, "dtype": "float32", "weights": "int"},
        # the King's subgraph configuration, Int32 weights in 1..100
        {"name": "ksg40_sc25_i32", "kind": "contract", "graph": "ksg", "n": 40, "gseed": 3,
         "sc": 25, "trials": 10, "dtype": "int32", "weights": "int"},
        # the headline workload: 3-regular n=300 seed 2 sliced to sc 25
        {"name": "slices_n300_sc25", "kind": "contract", "graph": "regular", "n": 300,
         "gseed": 2, "sc": 25, "trials": 200, "dtype": "float32", "weights": "unit"},
        # a burst of requests of the serving configuration, served to the end
        {"name": "serve_burst", "kind": "serve", "count": 16, "gseed": 5, "max_n": 160},
        # the branching tables of one branching step's candidate regions
        {"name": "tables_8x14", "kind": "tables", "n": 200, "gseed": 0, "regions": 8,
         "size": 14, "dtype": "float32", "weights": "unit"},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "solve", "contract", "contract", "contract",
                       "serve", "tables"])
    dtype = rng.choice(["float32", "int32"])
    weights = rng.choice(["int", "unit"])
    gseed = rng.randrange(1 << 30)
    if kind == "gemm":
        # each extent in 2^4 .. 2^12; a third of the draws all multiples of 16
        dims = [_log_int(rng, 16, 4096) for _ in range(3)]
        if rng.random() < 1 / 3:
            dims = [max(16, d // 16 * 16) for d in dims]
        M, N, K = dims
        batch = min(_log_int(rng, 1, 16), max(1, 4096 ** 3 // (M * N * K)))
        return {"kind": kind, "M": M, "N": N, "K": K, "batch": batch, "dtype": dtype}
    if kind == "serve":
        return {"kind": kind, "count": rng.randint(4, 16), "gseed": gseed,
                "max_n": rng.randint(110, 160)}
    if kind == "tables":
        return {"kind": kind, "n": 2 * rng.randint(40, 100), "gseed": gseed,
                "regions": rng.randint(1, 8), "size": rng.randint(8, 14), "dtype": dtype,
                "weights": weights}
    while True:
        case = {"kind": kind, "graph": "regular", "n": 0, "gseed": gseed, "sc": 0, "trials": 10,
                "dtype": dtype, "weights": weights}
        if kind == "solve":
            case.update(n=2 * rng.randint(30, 70), sc=rng.randint(12, 20))
        else:
            g = case["graph"] = rng.choice(["regular", "regular", "regular", "er", "ksg"])
            case["n"] = (2 * rng.randint(40, 125) if g == "regular" else
                         rng.randint(150, 250) if g == "er" else rng.randint(20, 40))
            case["sc"] = rng.randint(10, 25)
        try:
            macs = _macs(slices(case))
        except RuntimeError:  # more than MAX_SLICES
            macs = math.inf
        # (an Erdos-Renyi graph may kernelize away: nothing left to contract)
        if 0 < macs <= 2.0 ** MAX_LOG2_MACS:
            return case
        case["gseed"] = gseed = rng.randrange(1 << 30)


# ------------------------------------------------------------ the inputs ---
def _graph(kind, n, gseed):
    tb = package()
    if kind == "regular":
        return tb.random_regular_graph(n, 3, seed=gseed)
    if kind == "er":
        return tb.erdos_renyi(n, 3.0 / (n - 1), seed=gseed)
    return tb.random_ksg(n, n, 0.8, seed=gseed)


@functools.lru_cache(64)
def _slices(kind, n, gseed, sc, trials):
    tb = package()
    return tb.slice_graph(_graph(kind, n, gseed), None,
                          tb.ContractionTreeSlicer(sc_target=sc, order_trials=trials),
                          seed=gseed, max_slices=MAX_SLICES)


def slices(case):
    """The case's slices; a `solve` case is its largest one."""
    br = _slices(case["graph"], case["n"], case["gseed"], case["sc"], case["trials"])
    if case["kind"] == "solve":
        live = [b for b in br if b.code is not None]
        br = [max(live, key=lambda b: package().complexity(b).tc)] if live else []
    return br


def _macs(br):
    return sum(2.0 ** package().complexity(b).tc for b in br if b.code is not None)


def _weighted(br, dtype, weights, rng):
    """The slices with weights (1..100, or all 1) and fixed weights r from
    the random generator."""
    tb = package()
    out = []
    for b in br:
        w = rng.integers(1, 101, b.p.g.nv).astype(dtype) if weights == "int" else None
        out.append(tb.SlicedBranch(tb.MISProblem(b.p.g, w), b.code, int(rng.integers(0, 50))))
    return out


@functools.lru_cache(64)
def _requests(count, gseed, max_n):
    """Requests of the serving configuration: 3-regular and Erdos-Renyi
    graphs, sc_target 15..20, Float32 unit weights or Int32 weights."""
    rng = random.Random(gseed)
    out = []
    while len(out) < count:
        kind = rng.choice(["regular", "er"])
        n = 2 * rng.randint(50, max_n // 2) if kind == "regular" else rng.randint(100, 250)
        seed, sc = rng.randrange(1 << 30), rng.randint(15, 20)
        dtype, weights = rng.choice([("float32", "unit"), ("int32", "int")])
        br = _slices(kind, n, seed, sc, 10)
        if 0 < _macs(br) <= 2.0 ** 32:
            out.append((br, dtype, weights))
    return out


@functools.lru_cache(64)
def _regions(n, gseed, regions, size):
    tb = package()
    g = tb.random_regular_graph(n, 3, seed=gseed)
    rng = random.Random(gseed)
    return g, [tb.neighbor_region(g, [rng.randrange(n)], size) for _ in range(regions)]


def _gemm_inputs(case, seed):
    """A and B of mul!: integer values in [0, 2^10], a tenth of them the
    tropical zero; column-major, i.e. torch (batch, K, M) and (batch, N, K)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    f32 = case["dtype"] == "float32"
    out = []
    for shape in ((case["batch"], case["K"], case["M"]), (case["batch"], case["N"], case["K"])):
        x = torch.randint(0, 1025, shape, generator=gen, device="cuda", dtype=torch.int32)
        zero = torch.rand(shape, generator=gen, device="cuda") < 0.1
        x = x.to(torch.float32) if f32 else x
        x[zero] = -math.inf if f32 else I32_ZERO
        out.append(x if case["batch"] > 1 else x[0])
    return out


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "gemm":
        state["backend"] = backend()
        state["A"], state["B"] = _gemm_inputs(case, seed)
        return state
    rng = np.random.default_rng(seed)
    if kind == "serve":
        state["server"] = server()
        state["requests"] = [(_weighted(br, dtype, weights, rng), np.dtype(dtype))
                             for br, dtype, weights in
                             _requests(case["count"], case["gseed"], case["max_n"])]
        return state
    state["backend"] = backend()
    dtype = state["dtype"] = np.dtype(case["dtype"])
    if kind == "tables":
        tb = package()
        g, regions = _regions(case["n"], case["gseed"], case["regions"], case["size"])
        # each region's vertices in an order of their own, and weights
        regions = [[r[int(k)] for k in rng.permutation(len(r))] for r in regions]
        p = tb.MISProblem(g, rng.integers(1, 101, g.nv).astype(dtype)
                          if case["weights"] == "int" else None)
        state["items"] = [(p, r) for r in regions]
    else:
        state["branches"] = _weighted(slices(case), dtype, case["weights"], rng)
    return state


def run(state):
    kind = state["case"]["kind"]
    if kind == "gemm":
        return state["backend"].maxplus_gemm(state["A"], state["B"])
    if kind == "serve":
        srv = state["server"]
        tickets = [srv.submit(br, dtype) for br, dtype in state["requests"]]
        return [srv.wait(t) for t in tickets]
    if kind == "tables":
        tables = package().branching_tables(state["items"], state["dtype"],
                                            backend=state["backend"])
        # every region's alpha tensor, end to end, and which of its
        # configurations are rows
        rows = np.zeros((len(tables), 1 << state["case"]["size"]), np.uint8)
        for i, t in enumerate(tables):
            for row in t.table:
                rows[i, row] = 1
        return [np.concatenate([t.alpha for t in tables]), rows]
    if kind == "solve":
        return package().solve_slice(state["branches"][0], state["dtype"],
                                     backend=state["backend"])
    return package().contract_slices(state["branches"], state["dtype"],
                                     backend=state["backend"])


# -------------------------------------------------- what a pass must do ---
def _slice_bytes(br):
    n = 0
    for b in br:
        if b.code is not None:
            n += b.code.ix_ptr.nbytes + b.code.ix.nbytes + b.code.tree.nbytes
            n += 4 * b.p.g.nv
        n += 8 + 4  # r in, the result out
    return n


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        M, N, K, batch = case["M"], case["N"], case["K"], case["batch"]
        return {"bytes": 4 * batch * (M * K + K * N + M * N), "flops": 2 * batch * M * N * K}
    if kind == "serve":
        reqs = _requests(case["count"], case["gseed"], case["max_n"])
        return {"bytes": sum(_slice_bytes(br) for br, _, _ in reqs),
                "flops": 2 * sum(_macs(br) for br, _, _ in reqs)}
    if kind == "tables":
        # a region's configurations, each weighed once
        return {"bytes": 4 * case["regions"] * (1 << case["size"]),
                "flops": 2 * case["regions"] * case["size"] * (1 << case["size"])}
    br = slices(case)
    return {"bytes": _slice_bytes(br), "flops": 2 * _macs(br)}


# ------------------------------------------------- the results, 64 bits ---
def _canon(x, dtype):
    """The tropical zero as the element type writes it."""
    if np.dtype(dtype) == np.float32:
        return x
    return torch.where(x < -(1 << 29), torch.full_like(x, I32_ZERO), x)


def _exact_gemm(case, seed):
    A, B = (x.double() for x in _gemm_inputs(case, seed))
    A, B = (x if x.dim() == 3 else x[None] for x in (A, B))  # (b, K, M), (b, N, K)
    C = torch.full((A.shape[0], B.shape[1], A.shape[2]), -math.inf, dtype=torch.float64,
                   device=A.device)
    for k in range(A.shape[1]):
        torch.maximum(C, A[:, k, None, :] + B[:, :, k, None], out=C)
    C = _canon(C, case["dtype"])
    return C if case["batch"] > 1 else C[0]


def _exact_slice(b, r):
    """The tree's contraction in Float64: every node maxes A + B over the
    labels that occur nowhere else.  On the CPU (torch's GPU kernels take 16
    dimensions at most)."""
    if b.code is None:
        return float(r)
    ixs = b.code.ixs
    left = {}
    for ix in ixs:
        for l in ix:
            left[l] = left.get(l, 0) + 1
    w = np.ones(b.p.g.nv) if b.p.weights is None else np.asarray(b.p.weights, np.float64)
    edge = torch.tensor([[0.0, 0.0], [0.0, -math.inf]], dtype=torch.float64)
    vert = torch.zeros((b.p.g.nv, 2), dtype=torch.float64)
    vert[:, 1] = torch.as_tensor(w)
    nodes = [(list(ix), vert[ix[0]] if len(ix) == 1 else edge, {l: 1 for l in ix}) for ix in ixs]
    for j in range(len(b.code.tree) // 2):
        (la, A, ca), (lb, B, cb) = (nodes[int(c)] for c in b.code.tree[2 * j:2 * j + 2])
        cnt = dict(ca)
        for l, c in cb.items():
            cnt[l] = cnt.get(l, 0) + c
        drop = [l for l in cnt if cnt[l] == left[l]]
        keep = [l for l in cnt if cnt[l] != left[l]]
        order = keep + drop
        A = A.permute([la.index(l) for l in order if l in ca]).reshape(
            [2 if l in ca else 1 for l in order])
        B = B.permute([lb.index(l) for l in order if l in cb]).reshape(
            [2 if l in cb else 1 for l in order])
        C = A + B
        if drop:
            C = C.reshape(1 << len(keep), 1 << len(drop)).amax(1).reshape([2] * len(keep))
        nodes.append((keep, C, {l: cnt[l] for l in keep}))
    return float(nodes[-1][1]) + r


def _exact_ok(br):
    cs = [package().complexity(b) for b in br if b.code is not None]
    return len(br) <= 64 and all(c.sc <= 16 and c.tc <= 22 for c in cs)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        return _exact_gemm(case, seed)
    if kind == "tables":
        return None  # whole numbers
    rng = np.random.default_rng(seed)
    if kind == "serve":
        out = []
        for br, dtype, weights in _requests(case["count"], case["gseed"], case["max_n"]):
            br = _weighted(br, dtype, weights, rng)
            out.append(max(_exact_slice(b, b.r) for b in br) if _exact_ok(br) and len(br) <= 4
                       else None)
        return out
    br = _weighted(slices(case), np.dtype(case["dtype"]), case["weights"], rng)
    if not _exact_ok(br):
        return None
    if kind == "solve":
        return _exact_slice(br[0], 0.0)
    return np.array([_exact_slice(b, float(b.r)) for b in br])
