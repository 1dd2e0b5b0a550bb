"""Single-source frontiers at the sizes where the compaction, the work tables and the small-frontier
path change form, against the oracle (exact)."""
import numpy as np
import pytest

from conftest import random_csr

pytestmark = pytest.mark.gpu


def _csr(src, dst, w, n):
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, np.int64)
    np.add.at(row, np.asarray(src) + 1, 1)
    return (np.cumsum(row).astype(np.int32), np.asarray(dst)[order].astype(np.int32),
            np.asarray(w)[order].astype(np.int32))


def _check(npa, ctx, orc, row, col, w, src, scheds):
    G = npa.Graph.from_csr(ctx, row, col, w)
    ref, lev = orc.dijkstra(row, col, w, src)[0], orc.bfs_levels(row, col, src)
    for sch in scheds:
        d, st = ctx.sssp(G, src, sch)
        assert np.array_equal(d, ref), sch
        d, st = ctx.bfs(G, src, sch)
        assert np.array_equal(d, lev), sch
    G.free()


def _scheds(npa, delta=0):
    return [npa.Sched(level=lv, log2_t_lo=lo, log2_t_hi=hi, drive=dr, delta=delta)
            for lv, lo, hi in ((0, 4, 4), (1, 6, 6), (2, 2, 8)) for dr in (0, 1, 2)]


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 255, 1023, 1025, 2047, 8191, 8193, 70001])
def test_vertex_counts(npa, ctx, orc, n):
    """Bitmap words and tiles at their edges, dense and sparse frontiers, with and without a window."""
    rng = np.random.default_rng(n)
    row, col, w = random_csr(rng, n, 6 * n, 0, 40)
    src = int(rng.integers(n))
    _check(npa, ctx, orc, row, col, w, src, _scheds(npa) + _scheds(npa, 7))


@pytest.mark.parametrize("deg", [1, 3, 4, 7, 8, 9, 15, 16, 31, 63, 64, 65, 511, 513])
def test_one_degree(npa, ctx, orc, deg):
    """Every vertex in one out-degree class: below, at and above the serial rows, lane tiles of every
    width and the wavefront, workgroup and grid bins."""
    rng = np.random.default_rng(1000 + deg)
    n = 3000 if deg > 60 else 20000
    row = (np.arange(n + 1) * deg).astype(np.int32)
    col = rng.integers(0, n, n * deg).astype(np.int32)
    w = rng.integers(1, 100, n * deg).astype(np.int32)
    _check(npa, ctx, orc, row, col, w, 5, _scheds(npa))


@pytest.mark.parametrize("width", [1, 2, 255, 256, 511, 512, 513, 700, 2000])
@pytest.mark.parametrize("fan", [1, 4, 8, 9])
def test_layers_of_one_width(npa, ctx, orc, width, fan):
    """A ladder of layers: every frontier has `width` vertices and width x fan edges, below, at and
    above what one workgroup takes alone, for more layers than one visit runs."""
    rng = np.random.default_rng(width * 10 + fan)
    layers = 600 if width <= 2 else 12
    n = 1 + width * layers
    src, dst = [np.zeros(width, np.int64)], [1 + np.arange(width)]
    for k in range(layers - 1):
        a = 1 + width * k + np.repeat(np.arange(width), fan)
        b = 1 + width * (k + 1) + rng.integers(0, width, width * fan)
        b[::fan] = 1 + width * (k + 1) + np.arange(width)     # every vertex of the next layer is reached
        src.append(a)
        dst.append(b)
    src, dst = np.concatenate(src), np.concatenate(dst)
    row, col, w = _csr(src, dst, rng.integers(1, 50, len(src)), n)
    _check(npa, ctx, orc, row, col, w, 0, [npa.Sched(level=lv, drive=dr) for lv in (1, 2) for dr in (0, 2)])


def test_small_and_large_frontiers_alternate(npa, ctx, orc):
    """One vertex -> 3,000 -> one -> 3,000 ...: the small-frontier path is entered and left again and
    again, overflows its list, and vertices without out-edges appear in both."""
    rng = np.random.default_rng(9)
    src, dst, at = [], [], 0
    for k in range(8):
        wide = 3000 if k % 2 == 0 else 600
        src += [np.full(wide, at), at + 1 + np.arange(wide - 100)]
        dst += [at + 1 + np.arange(wide), np.full(wide - 100, at + 1 + wide)]   # 100 dead ends per layer
        at += 1 + wide
    src, dst = np.concatenate(src), np.concatenate(dst)
    row, col, w = _csr(src, dst, rng.integers(1, 30, len(src)), at + 1)
    _check(npa, ctx, orc, row, col, w, 0, _scheds(npa))


@pytest.mark.parametrize("cap", [1, 2, 37, 255, 256, 257, 400])
def test_iteration_cap_inside_small_frontiers(npa, ctx, orc, cap):
    """max_iters stops a chain of one-vertex frontiers after exactly that many expansions."""
    n = 500
    row = np.minimum(np.arange(n + 1), n - 1).astype(np.int32)
    G = npa.Graph.from_csr(ctx, row, np.arange(1, n, dtype=np.int32), np.ones(n - 1, np.int32))
    buf = npa.DeviceBuffer(ctx, n)
    with pytest.raises(npa.NpError):
        ctx.sssp_device(G, 0, buf.ptr, npa.Sched(level=1, max_iters=cap))
    assert int((buf.to_host() < npa.INF).sum()) == cap + 1
    d, st = ctx.sssp(G, 0, npa.Sched(level=1))
    assert np.array_equal(d, np.arange(n)) and st.iterations == n - 1
    buf.free()
    G.free()


def test_concatenated_small_frontiers(npa, ctx, orc):
    """Instances of several graphs in one slot space, from one-vertex frontiers to the last."""
    rng = np.random.default_rng(11)
    graphs = [npa.Graph.from_csr(ctx, *random_csr(rng, n, 3 * n, 1, 20)) for n in (1, 3, 40, 1024, 1025, 5000)]
    srcs = [int(rng.integers(g.n)) for g in graphs]
    for unit in (False, True):
        b = npa.Batch(ctx, graphs, srcs, unit=unit)
        for dr in (0, 1, 2):
            b.solve(npa.Sched(level=2, log2_t_lo=4, log2_t_hi=8, drive=dr))
            for i, (g, s) in enumerate(zip(graphs, srcs)):
                row, col, w = g.download()
                ref = orc.bfs_levels(row, col, s) if unit else orc.dijkstra(row, col, w, s)[0]
                assert np.array_equal(b.get(i), ref), (unit, dr, i)
        b.free()
    for g in graphs:
        g.free()


@pytest.mark.parametrize("deg", [32767, 32768, 32769, 65537, 100000])
def test_rows_longer_than_a_workgroup_chunk(npa, ctx, orc, deg):
    """Block level: rows just below, at and above the chunk, and of several chunks, reached first,
    later and again; both frontier kinds and every drive."""
    rng = np.random.default_rng(deg)
    n = 4000
    src = np.concatenate([np.zeros(deg, np.int64), np.full(deg - 1, 7), rng.integers(0, n, 3 * n)])
    dst = rng.integers(0, n, len(src))
    row, col, w = _csr(src, dst, rng.integers(1, 200, len(src)), n)
    _check(npa, ctx, orc, row, col, w, 5, [npa.Sched(level=1, drive=dr, frontier=fr) for dr in (0, 1, 2) for fr in (0, 1)])


@pytest.mark.parametrize("nsrc", [2, 3, 8, 17, 32])
@pytest.mark.parametrize("kind", ["grid", "rmat", "dead_ends"])
def test_packed_window_moves_deferred_pairs(npa, ctx, orc, kind, nsrc):
    """Windowed packs: pairs deferred, flagged again below and above the window, taken when it
    rises; from a window that defers nearly everything to one that ends at its first rise and one
    whose first rise would pass the largest threshold; repeated solves on one batch, with solves
    without a window between."""
    rng = np.random.default_rng(nsrc)
    if kind == "grid":
        G = npa.Graph.grid(ctx, 40, 53, None, 1, 255, seed=61)
    elif kind == "rmat":
        G = npa.Graph.rmat(ctx, 11, 8, wmin=1, wmax=255, seed=62)
    else:                                   # vertices without out-edges, zero weights, unreached vertices
        row, col, w = random_csr(rng, 1500, 4000, 0, 300)
        G = npa.Graph.from_csr(ctx, row, col, w)
    row, col, w = G.download()
    srcs = [int(s) for s in rng.integers(0, G.n, nsrc)]
    ref = [orc.dijkstra(row, col, w, s)[0] for s in srcs]
    b = npa.Batch(ctx, [G] * nsrc, srcs)
    for dr in (0, 1, 2):
        for delta in (1, 40, 0, 700, 2 ** 30):
            b.solve(npa.Sched(level=2, log2_t_lo=3, log2_t_hi=7, drive=dr, delta=delta))
            for i in range(nsrc):
                assert np.array_equal(b.get(i), ref[i]), (dr, delta, i)
    b.free()
    G.free()


@pytest.mark.parametrize("n", [3, 4, 5, 6, 7, 8, 1027, 4099, 70001])
def test_distance_range_is_checked_at_every_index(npa, ctx, n):
    """src -> a -> b with 2^29 on both edges: b's distance would be 2^30, which is refused wherever a
    (the only finite distance near the limit) lies in the buffer, also one that is not aligned to 16
    bytes; one less and it is accepted."""
    half = 1 << 29
    buf = npa.DeviceBuffer(ctx, n + 3)
    for a in sorted({0, 1, 2, 3, n // 2, n - 3, n - 2, n - 1} & set(range(n))):
        src, b = [v for v in (0, 1, n - 1, n // 2) if v != a][:2]
        for last, fits in ((half, False), (half - 1, True)):
            G = npa.Graph.from_csr(ctx, *_csr([src, a], [a, b], [half, last], n))
            want = np.full(n, npa.INF, np.int32)
            want[src], want[a], want[b] = 0, half, half + last
            for off in range(4):
                if fits:
                    ctx.sssp_device(G, src, buf.ptr + 4 * off, npa.Sched(level=1))
                    assert np.array_equal(buf.to_host()[off:off + n], want), (a, off)
                else:
                    with pytest.raises(npa.NpError):
                        ctx.sssp_device(G, src, buf.ptr + 4 * off, npa.Sched(level=1))
            G.free()
    buf.free()


@pytest.mark.parametrize("nsrc", [2, 3, 16])
def test_packed_window_follows_the_current_distances_on_every_drive(npa, ctx, nsrc):
    """One launch per solve sees other workgroups' distances as launches per step do: a window that
    goes by rows of earlier iterations defers pairs below it and rises above them, which showed as more
    than twice the iterations."""
    G = npa.Graph.grid(ctx, 700, 701, None, 1, 1000, seed=97)
    srcs = [int(s) for s in npa.pick_sources(G.download()[0], nsrc, 9)]
    b = npa.Batch(ctx, [G] * nsrc, srcs)
    for delta in (1000, 3000, 8000):
        it = [b.solve(npa.Sched(level=2, log2_t_lo=6, log2_t_hi=8, delta=delta, drive=dr)).iterations for dr in (0, 1, 2)]
        assert it[0] <= 1.15 * min(it[1:]), (delta, it)
    b.free()
    G.free()
