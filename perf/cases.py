"""The work this framework is used for, as cases that can be timed and compared.

A case is a dict of plain values; `prepare` makes what a program holds before the call (the graph on the
device, its sources, result buffers, a batch), `run` makes one pass through the public entry points of the
Python package, `work` counts what a pass cannot do without, and `exact` gives floating results in 64 bits.

Kinds and what they stand for:
  sssp      one shortest-path solve (SSSP_GPU), plain or learned schedule, result on the host or the device
  bfs       one level solve (BFS_REC_GPU)
  batch     many sources and graphs solved together: source-packed, priority window, small graphs concatenated
  bc        betweenness centrality over a set of sources (BC_GPU; forward counts and backward sums)
  color     graph coloring (GRAPH_COLOR_GPU)
  pagerank  ranks to convergence (PAGERANK_GPU), in-edge lists built in the call
  spmv      float64 matrix-vector product on host vectors (SpMV_GPU)
Graphs: R-MAT (a, b, c = .57, .19, .19, ids permuted), uniform random (er), and grids with 1 % long-range edges.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEV = "cuda"
_ctx = None


def _package():
    """The package's folder name has a hyphen, so it is loaded from its file."""
    name = "nested_parallelism_amd"
    if name not in sys.modules:
        folder = os.path.join(ROOT, "nested-parallelism_amd")
        spec = importlib.util.spec_from_file_location(name, os.path.join(folder, "__init__.py"),
                                                      submodule_search_locations=[folder])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def _context():
    """One context for the program, as a user's program has."""
    global _ctx
    if _ctx is None:
        _ctx = _package().Context(0)
    return _ctx


# ---------------------------------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------------------------------
def listed():
    return [
        # one query on a small graph, result on the host: latency and launches
        dict(name="sssp_er_64k", kind="sssp", graph="er", n=65536, m=1048576, wmax=100, level=1, lo=6, hi=6, drive=0,
             frontier=0, host=True),
        # one query on a skewed graph with the default (block-level) schedule, result kept on the device
        dict(name="sssp_rmat_4m", kind="sssp", graph="rmat", n=4194304, m=67108864, wmax=255, level=1, lo=6, hi=6,
             drive=0, frontier=0, host=False),
        # one query on a road-like graph: many small iterations
        dict(name="sssp_grid_2k", kind="sssp", graph="grid", n=2048 * 2048, m=0, rows=2048, cols=2048, wmax=1000,
             level=1, lo=6, hi=6, drive=0, frontier=0, host=False),
        # levels from one source, a vertex count that is no power of two
        dict(name="bfs_rmat_3m", kind="bfs", graph="rmat", n=3000017, m=48000271, wmax=255, level=2, lo=6, hi=6,
             drive=0, frontier=0, host=False),
        # the largest: 16 sources of one graph of 16.8 M vertices and 268 M edges, source-packed
        dict(name="batch_rmat_16m_16src", kind="batch", unit=False, graph="rmat", n=16777216, m=268435456, wmax=255,
             sources=16, small=0, level=2, lo=4, hi=10, drive=2, delta=0, hold=10),
        # 32 sources of a road-like graph with a priority window
        dict(name="batch_grid_2k_32src", kind="batch", unit=False, graph="grid", n=2048 * 2048, m=0, rows=2048,
             cols=2048, wmax=1000, sources=32, small=0, level=2, lo=6, hi=8, drive=2, delta=4004, hold=0),
        # 16 sources of one graph together with 40 small graphs of one source each
        dict(name="batch_mixed_40", kind="batch", unit=False, graph="rmat", n=262144, m=4194304, wmax=255, sources=16,
             small=40, level=2, lo=4, hi=10, drive=2, delta=0, hold=0),
        # levels from 16 sources together
        dict(name="batch_bfs_4m_16src", kind="batch", unit=True, graph="rmat", n=4194304, m=67108864, wmax=255,
             sources=16, small=0, level=2, lo=4, hi=10, drive=2, delta=0, hold=10),
        # centrality from 256 sources: forward path counts and backward dependencies
        dict(name="bc_rmat_64k_256src", kind="bc", graph="rmat", n=65536, m=1048576, wmax=255, sources=256),
        # a whole coloring, result on the host
        dict(name="color_rmat_1m", kind="color", graph="rmat", n=1048576, m=16777216, wmax=255),
        # ranks of a whole graph to convergence
        dict(name="pagerank_rmat_1m", kind="pagerank", graph="rmat", n=1048576, m=16777216, wmax=255),
        # one product with values and vector on the host
        dict(name="spmv_rmat_1m", kind="spmv", graph="rmat", n=1048576, m=16777216, wmax=255),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_graph(rng, kinds, n_lo, n_hi):
    graph = rng.choice(kinds)
    n = _log_int(rng, n_lo, n_hi)
    if graph == "grid":
        rows = max(2, int(math.sqrt(n) * rng.uniform(0.5, 2.0)))
        cols = max(2, n // rows)
        return dict(graph="grid", n=rows * cols, m=0, rows=rows, cols=cols, wmax=1000)
    return dict(graph=graph, n=n, m=int(n * rng.uniform(4.0, 16.0)), wmax=rng.choice([100, 255]))


def draw(rng):
    kind = rng.choice(["sssp", "sssp", "bfs", "batch", "batch", "bc", "color", "pagerank", "spmv"])
    if kind in ("sssp", "bfs"):
        g = _draw_graph(rng, ["er", "rmat", "grid"], 1000, 4194304)
        sched = rng.choice([dict(level=0, lo=6, hi=6), dict(level=1, lo=6, hi=6), dict(level=2, lo=6, hi=6),
                            dict(level=2, lo=4, hi=10), dict(level=-1, lo=6, hi=12)])
        return dict(kind=kind, **g, **sched, drive=rng.choice([0, 0, 2]), frontier=rng.choice([0, 0, 0, 1]),
                    host=g["n"] <= 200000)
    if kind == "batch":
        g = _draw_graph(rng, ["er", "rmat", "grid"], 2000, 2097152)
        unit = rng.random() < 0.35
        grid = g["graph"] == "grid"
        return dict(kind="batch", unit=unit, **g, sources=rng.randint(2, 32), small=rng.choice([0, 0, 7, 24]), level=2,
                    lo=6 if grid else 4, hi=8 if grid else 10, drive=rng.choice([0, 2, 2]),
                    delta=4004 if grid and not unit else 0, hold=0 if grid else rng.choice([0, 10]))
    if kind == "bc":
        g = _draw_graph(rng, ["er", "rmat"], 1000, 131072)
        return dict(kind="bc", **g, sources=rng.randint(1, 256))
    if kind == "color":
        return dict(kind="color", **_draw_graph(rng, ["er", "rmat", "grid"], 1000, 1048576))
    g = _draw_graph(rng, ["er", "rmat"], 1000, 1048576)
    return dict(kind=kind, **g)


# ---------------------------------------------------------------------------------------------------
# graphs, as device CSR arrays
# ---------------------------------------------------------------------------------------------------
def _rmat_edges(n, m, g):
    """m edges among n vertices: R-MAT over the next power of two, ids permuted, edges that leave [0, n) replaced
    by ones folded back into it."""
    scale = max(1, (n - 1).bit_length())
    src = torch.zeros(m, dtype=torch.int32, device=DEV)
    dst = torch.zeros(m, dtype=torch.int32, device=DEV)
    for _ in range(scale):
        r = torch.rand(m, device=DEV, generator=g)
        src.mul_(2).add_(r >= 0.76)
        dst.mul_(2).add_(((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    perm = torch.randperm(1 << scale, device=DEV, generator=g, dtype=torch.int32)
    src, dst = perm[src], perm[dst]
    if n != 1 << scale:
        src.remainder_(n)
        dst.remainder_(n)
    return src, dst


def _grid_edges(rows, cols, g):
    v = torch.arange(rows * cols, dtype=torch.int32, device=DEV).view(rows, cols)
    a = torch.cat([v[:, :-1].reshape(-1), v[:-1, :].reshape(-1)])
    b = torch.cat([v[:, 1:].reshape(-1), v[1:, :].reshape(-1)])
    far = 2 * a.numel() // 100
    fs = torch.randint(0, rows * cols, (far,), device=DEV, generator=g, dtype=torch.int32)
    fd = torch.randint(0, rows * cols, (far,), device=DEV, generator=g, dtype=torch.int32)
    return torch.cat([a, b, fs]), torch.cat([b, a, fd])


def _csr(case, seed):
    """(row, col, w) int32 tensors on the device, from the seed alone."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    n = case["n"]
    if case["graph"] == "rmat":
        src, dst = _rmat_edges(n, case["m"], g)
    elif case["graph"] == "grid":
        src, dst = _grid_edges(case["rows"], case["cols"], g)
    else:
        src = torch.randint(0, n, (case["m"],), device=DEV, generator=g, dtype=torch.int32)
        dst = torch.randint(0, n, (case["m"],), device=DEV, generator=g, dtype=torch.int32)
    src, order = torch.sort(src, stable=True)
    col = dst[order]
    del order, dst
    row = torch.searchsorted(src, torch.arange(n + 1, device=DEV, dtype=torch.int32), out_int32=True)
    del src
    w = torch.randint(1, case["wmax"] + 1, (col.numel(),), device=DEV, generator=g, dtype=torch.int32)
    return row, col, w


def _sources(row, k, seed):
    """k different vertices with out-edges."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) + 77)
    live = torch.nonzero(row[1:] > row[:-1]).view(-1)
    pick = torch.randperm(live.numel(), device=DEV, generator=g)[:k]
    return [int(v) for v in live[pick].cpu()]


def _wrap(ctx, row, col, w):
    """np_graph over a program's own device arrays (the arrays have to outlive it)."""
    npa = _package()
    torch.cuda.synchronize()
    h = ctypes.c_void_p()
    rc = npa.load().np_graph_wrap_device(ctx.h, row.numel() - 1, col.numel(), ctypes.c_void_p(row.data_ptr()),
                                         ctypes.c_void_p(col.data_ptr()), ctypes.c_void_p(w.data_ptr()), ctypes.byref(h))
    if rc:
        raise npa.NpError(rc, npa.last_error())
    return npa.Graph(ctx, h)


class _Held:
    """A device array of the library, for torch (it stays the library's)."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<i4", data=(ptr, False), strides=None, version=2)


# ---------------------------------------------------------------------------------------------------
# one case
# ---------------------------------------------------------------------------------------------------
def prepare(case, seed):
    npa, ctx = _package(), _context()
    row, col, w = _csr(case, seed)
    graph = _wrap(ctx, row, col, w)
    state = dict(case=case, ctx=ctx, graph=graph, keep=[row, col, w])
    kind = case["kind"]
    if kind in ("sssp", "bfs"):
        state["src"] = _sources(row, 1, seed)[0]
        state["sched"] = npa.Sched(level=case["level"], log2_t_lo=case["lo"], log2_t_hi=case["hi"], drive=case["drive"],
                                   frontier=case["frontier"])
        if case["level"] == npa.LEVEL_LEARNED:
            ctx.model_set(np.fromfile(os.path.join(ROOT, "nested-parallelism_amd", "sched_mlp.f32"), np.float32))
        if not case["host"]:
            state["out"] = torch.empty(case["n"], dtype=torch.int32, device=DEV)
    elif kind == "batch":
        graphs, srcs = [graph] * case["sources"], _sources(row, case["sources"], seed)
        graphs = graphs[:len(srcs)]
        for i in range(case["small"]):
            n = 1 << (12 + i % 5)
            one = dict(graph="rmat", n=n, m=16 * n, wmax=255)
            r, c, x = _csr(one, seed + 1000 * (i + 1))
            graphs.append(_wrap(ctx, r, c, x))
            srcs += _sources(r, 1, seed + i)
            state["keep"] += [r, c, x]
        state["batch"] = npa.Batch(ctx, graphs, srcs, unit=case["unit"])
        state["views"] = {}
        state["sched"] = npa.Sched(level=case["level"], log2_t_lo=case["lo"], log2_t_hi=case["hi"], drive=case["drive"],
                                   delta=case["delta"], pack_hold=case["hold"])
    elif kind == "bc":
        state["srcs"] = _sources(row, case["sources"], seed)
    elif kind == "spmv":
        rng = np.random.default_rng(seed)
        state["data"] = rng.standard_normal(graph.m)
        state["x"] = rng.standard_normal(graph.n)
    torch.cuda.synchronize()
    return state


def run(state):
    case, ctx, graph = state["case"], state["ctx"], state["graph"]
    kind = case["kind"]
    if kind == "sssp":
        if case["host"]:
            return ctx.sssp(graph, state["src"], state["sched"])[0]
        ctx.sssp_device(graph, state["src"], state["out"].data_ptr(), state["sched"])
        return state["out"]
    if kind == "bfs":
        if case["host"]:
            return ctx.bfs(graph, state["src"], state["sched"])[0]
        ctx.bfs_device(graph, state["src"], state["out"].data_ptr(), state["sched"])
        return state["out"]
    if kind == "batch":
        b, views, got = state["batch"], state["views"], []
        b.solve(state["sched"])
        for i in range(b.count):
            p = b.device_dist(i)
            if p not in views:
                views[p] = torch.as_tensor(_Held(p, b.graphs[i].n), device=DEV)
                views[p].owner = (b, state["keep"])  # the memory is the batch's: it lives as long as a view does
            got.append(views[p])
        return got
    if kind == "bc":
        return ctx.bc(graph, state["srcs"])[0]
    if kind == "color":
        return ctx.color(graph)[0]
    if kind == "pagerank":
        return ctx.pagerank(graph)[0]
    return ctx.spmv(graph, state["data"], state["x"])[0]


def _edges(case):
    if case["graph"] != "grid":
        return case["m"]
    r, c = case["rows"], case["cols"]
    e = 2 * (r * (c - 1) + c * (r - 1))
    return e + e // 100


def work(case):
    """Each input read once, each output written once; operations where the path computes with numbers."""
    n, m, kind = case["n"], _edges(case), case["kind"]
    offsets = 4 * (n + 1)
    if kind == "sssp":
        return dict(bytes=offsets + 8 * m + 4 * n, flops=m)
    if kind == "bfs":
        return dict(bytes=offsets + 4 * m + 4 * n, flops=m)
    if kind == "batch":
        k = case["sources"]
        sizes = [1 << (12 + i % 5) for i in range(case["small"])]
        per = 4 if case["unit"] else 8
        return dict(bytes=offsets + per * m + 4 * n * k + sum(4 * s + per * 16 * s + 4 * s for s in sizes),
                    flops=m * k + sum(16 * s for s in sizes))
    if kind == "bc":
        return dict(bytes=offsets + 4 * m + 4 * n, flops=4 * m * case["sources"])
    if kind == "color":
        return dict(bytes=offsets + 4 * m + 4 * n, flops=m)
    if kind == "pagerank":
        return dict(bytes=offsets + 4 * m + 4 * n, flops=2 * 24 * m)  # about 24 iterations
    return dict(bytes=offsets + 12 * m + 16 * n, flops=2 * m)


# ---------------------------------------------------------------------------------------------------
# floating results in 64 bits
# ---------------------------------------------------------------------------------------------------
def _exact_pagerank(n, src, dst, deg):
    rank = torch.full((n,), 1000.0 / n, dtype=torch.float64, device=DEV)
    inv = torch.where(deg > 0, 1.0 / deg.clamp(min=1), torch.zeros_like(rank))
    for _ in range(1000):
        new = torch.zeros_like(rank).index_add_(0, dst, (rank * inv)[src])
        new = 0.5 * new + 0.5 * 1000.0 / n + 0.5 * rank[deg == 0].sum() / n
        change = float((new - rank).abs().max())
        rank = new
        if not change > 1e-13:
            break
    return rank


def _exact_bc(n, src, dst, sources):
    total = torch.zeros(n, dtype=torch.float64, device=DEV)
    for at in range(0, len(sources), 16):
        some = torch.tensor(sources[at:at + 16], device=DEV)
        k = some.numel()
        lane = torch.arange(k, device=DEV)
        level = torch.full((n, k), -1, dtype=torch.int32, device=DEV)
        sigma = torch.zeros((n, k), dtype=torch.float64, device=DEV)
        level[some, lane] = 0
        sigma[some, lane] = 1.0
        depth = 0
        while True:
            flow = torch.where(level == depth, sigma, torch.zeros_like(sigma))
            got = torch.zeros_like(sigma).index_add_(0, dst, flow[src])
            fresh = (level < 0) & (got > 0)
            if not bool(fresh.any()):
                break
            depth += 1
            level[fresh] = depth
            sigma = torch.where(fresh, got, sigma)
        delta = torch.zeros_like(sigma)
        for d in range(depth - 1, -1, -1):
            part = torch.where(level == d + 1, (1.0 + delta) / sigma.clamp(min=1.0), torch.zeros_like(sigma))
            back = torch.zeros_like(sigma).index_add_(0, src, part[dst])
            delta = torch.where(level == d, sigma * back, delta)
        delta[some, lane] = 0.0
        total += delta.sum(1)
    return total


def exact(case, seed):
    """bc, pagerank and spmv compute floating numbers; every other result is whole numbers."""
    kind = case["kind"]
    if kind not in ("bc", "pagerank", "spmv"):
        return None
    row, col, _ = _csr(case, seed)
    n = case["n"]
    deg = (row[1:] - row[:-1]).long()
    src = torch.repeat_interleave(torch.arange(n, device=DEV), deg)
    dst = col.long()
    if kind == "pagerank":
        return _exact_pagerank(n, src, dst, deg.double())
    if kind == "bc":
        return _exact_bc(n, src, dst, _sources(row, case["sources"], seed))
    rng = np.random.default_rng(seed)
    data = torch.from_numpy(rng.standard_normal(col.numel())).to(DEV)
    x = torch.from_numpy(rng.standard_normal(n)).to(DEV)
    return torch.zeros(n, dtype=torch.float64, device=DEV).index_add_(0, src, data * x[dst])
