"""Results of a batch in original vertex ids: one launch per pack and one for the renumbered
concatenated instances, made at the first request after a solve; all against the oracle (exact)."""
import numpy as np
import pytest

from conftest import random_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("relabel", [0, 1])
@pytest.mark.parametrize("k", [2, 3, 4, 7, 8, 9, 16, 17, 31, 32])
def test_every_row_width_and_request_order(npa, ctx, orc, k, relabel):
    """Rows of 2..32 distances, full and partly used, vertex counts around a workgroup, requests in
    any order and repeated, and a second solve (other lengths) that replaces the first's results."""
    rng = np.random.default_rng(100 * k + relabel)
    ctx.set_option(npa.CTX_RELABEL, relabel)
    try:
        G = npa.Graph.from_csr(ctx, *random_csr(rng, 255 + k, 3000, 1, 50))
        small = [npa.Graph.from_csr(ctx, *random_csr(rng, n, 5 * n, 1, 50)) for n in (1, 255, 1025)]
    finally:
        ctx.set_option(npa.CTX_RELABEL, 2)
    graphs = [G] * k + small
    srcs = [int(s) for s in rng.permutation(G.n)[:k]] + [0, 254, 1024]
    order = rng.permutation(len(graphs))
    graphs, srcs = [graphs[i] for i in order], [srcs[i] for i in order]
    csr = {id(g): g.download() for g in [G] + small}
    ref = [orc.dijkstra(*csr[id(g)], s)[0] for g, s in zip(graphs, srcs)]
    b = npa.Batch(ctx, graphs, srcs)
    assert b.layout() == (1, 3)
    for sched in (npa.Sched(level=2, log2_t_lo=4, log2_t_hi=10), npa.Sched(level=1, drive=npa.DRIVE_GRAPH)):
        b.solve(sched)
        for i in list(rng.permutation(len(graphs))) + [0, 0]:
            assert np.array_equal(b.get(int(i)), ref[i]), (k, relabel, i)
    # a solve that stops after one expansion: its distances, not the ones unpacked before
    with pytest.raises(npa.NpError):
        b.solve(npa.Sched(level=1, max_iters=1))
    for i, (g, s) in enumerate(zip(graphs, srcs)):
        d = b.get(i)
        row, col, w = csr[id(g)]
        near = set(col[row[s]:row[s + 1]]) | {s}
        far = [v for v in range(g.n) if v not in near]
        if g is G:
            assert d[s] == 0 and (d[far] == npa.INF).all(), i
    b.free()
    for g in [G] + small:
        g.free()


@pytest.mark.parametrize("kind", ["rmat", "rmat_hold", "zero_weights", "large_weights", "too_large_weights",
                                  "cut_off_sources"])
@pytest.mark.parametrize("k", [3, 4, 5, 16, 31, 32])
def test_bound_filter_is_exact(npa, ctx, orc, k, kind):
    """Packs of a renumbered graph on the per-iteration drives drop edges by the vertices' bounds: row
    widths 4..32, rows in every class around the tile and grid bins, weights at the ends of the
    codes' range, and sources that never reach the hub (no part in the bounds)."""
    rng = np.random.default_rng(200 + k)
    ctx.set_option(npa.CTX_RELABEL, 1)
    wmax = {"zero_weights": 0, "large_weights": 1 << 22, "too_large_weights": 1 << 26}.get(kind, 255)
    try:
        g0 = npa.Graph.rmat(ctx, 12, 24, wmin=0 if wmax == 0 else 1, wmax=max(wmax, 1), seed=300 + k)
        row, col, w = g0.download()
        if kind == "zero_weights":
            w[:] = 0
        srcs = [int(s) for s in npa.pick_sources(row, k, 4)]
        if kind == "cut_off_sources":                 # a path that never enters the R-MAT part
            n = len(row) - 1
            row = np.concatenate([row, row[-1] + np.arange(1, 41)]).astype(np.int32)
            col = np.concatenate([col, n + np.minimum(np.arange(1, 41), 39)]).astype(np.int32)
            w = np.concatenate([w, rng.integers(1, 255, 40)]).astype(np.int32)
            srcs[0] = n + 3
            if k > 8:
                srcs[1] = n
        G = npa.Graph.from_csr(ctx, row, col, w)
    finally:
        ctx.set_option(npa.CTX_RELABEL, 2)
    b = npa.Batch(ctx, [G] * k, srcs)
    ref = [orc.dijkstra(row, col, w, s)[0] for s in srcs]
    hold = 6 if kind == "rmat_hold" else 0
    for level, lo, hi, drive in ((2, 4, 10, npa.DRIVE_GRAPH), (2, 4, 6, npa.DRIVE_HOSTLOOP), (1, 6, 6, npa.DRIVE_GRAPH),
                                 (0, 3, 3, npa.DRIVE_HOSTLOOP), (2, 6, 12, npa.DRIVE_PERSISTENT)):
        b.solve(npa.Sched(level=level, log2_t_lo=lo, log2_t_hi=hi, drive=drive, pack_hold=hold))
        for i in range(k):
            assert np.array_equal(b.get(i), ref[i]), (kind, k, level, drive, i)
    b.free()
    G.free()
    g0.free()


@pytest.mark.parametrize("unit", [False, True])
@pytest.mark.parametrize("n, hold", [(40, 6), (2100, 6), (9000, 7)])
def test_hold_with_hubs_side_by_side(npa, ctx, orc, n, hold, unit):
    """Every vertex is heavy enough to be held, in every word of a wavefront's share (more than one
    look at the rows per wavefront), with duplicate sources and vertices reached by few."""
    rng = np.random.default_rng(n + hold)
    deg = rng.integers(33, 140, n)
    row = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    col = rng.integers(0, n, row[-1]).astype(np.int32)
    w = rng.integers(1, 60, row[-1]).astype(np.int32)
    srcs = [int(s) for s in rng.integers(0, n, 19)] + [3, 3, 3]
    ctx.set_option(npa.CTX_RELABEL, 1)
    try:
        G = npa.Graph.from_csr(ctx, row, col, w)
    finally:
        ctx.set_option(npa.CTX_RELABEL, 2)
    b = npa.Batch(ctx, [G] * len(srcs), srcs, unit=unit)
    for drive in (0, 1, 2):
        b.solve(npa.Sched(level=2, log2_t_lo=4, log2_t_hi=6, drive=drive, pack_hold=hold))
        for i, s in enumerate(srcs):
            ref = orc.bfs_levels(row, col, s) if unit else orc.dijkstra(row, col, w, s)[0]
            assert np.array_equal(b.get(i), ref), (drive, i)
    b.free()
    G.free()


def _at(npa, ctx, ptr, n):
    out = np.empty(n, np.int32)
    assert npa.load().np_dev_copy(ctx.h, out.ctypes.data, ptr, out.nbytes, 1) == 0
    return out


@pytest.mark.parametrize("k", [2, 4, 9, 32])
@pytest.mark.parametrize("part", ["pack", "concatenated"])
def test_one_request_writes_one_result(npa, ctx, orc, k, part):
    """A program that asks for one result after each solve does not pay for the others: what an earlier
    solve wrote for another instance is still there.  Then every mix of requests over repeated solves
    of a pack, or of renumbered graphs in one slot space, gives the results of its own solve."""
    rng = np.random.default_rng(400 + k)
    ctx.set_option(npa.CTX_RELABEL, 1)
    try:
        graphs = [npa.Graph.from_csr(ctx, *random_csr(rng, 700 + 13 * j, 6000, 1, 50)) for j in range(1 if part == "pack" else k)]
    finally:
        ctx.set_option(npa.CTX_RELABEL, 2)
    of = graphs * k if part == "pack" else graphs
    host = [g.download() for g in graphs]
    csr = host * k if part == "pack" else host
    srcs = [int(np.argmax(np.diff(r[0]) == d)) for r, d in zip(csr, [max(np.diff(r[0])) for r in csr])]
    srcs = [int(rng.integers(g.n)) if part == "pack" and j else s for j, (g, s) in enumerate(zip(of, srcs))]
    full = [orc.dijkstra(*r, s)[0] for r, s in zip(csr, srcs)]
    b = npa.Batch(ctx, of, srcs)
    assert b.layout() == ((1, 0) if part == "pack" else (0, k))

    def solve(stop):
        """A whole solve, or one stopped after the sources' own expansion."""
        if not stop:
            b.solve(npa.Sched(level=1))
            return full
        with pytest.raises(npa.NpError):
            b.solve(npa.Sched(level=1, max_iters=1))
        one = []
        for (row, col, w), s, g in zip(csr, srcs, of):
            d = np.full(g.n, npa.INF, np.int32)
            np.minimum.at(d, col[row[s]:row[s + 1]], w[row[s]:row[s + 1]])
            d[s] = 0
            one.append(d)
        return one

    solve(False)
    p = b.device_dist(1)
    assert np.array_equal(_at(npa, ctx, p, of[1].n), full[1])
    want = solve(True)
    assert np.array_equal(_at(npa, ctx, b.device_dist(0), of[0].n), want[0])
    assert np.array_equal(_at(npa, ctx, p, of[1].n), full[1])
    for step, asked in enumerate([[0], [1], [0, 1], list(range(k)), [k - 1], [k - 1, 0], [0], list(range(k)), [], [1, 1, 0]]):
        want = solve(step % 2 == 1)
        for i in asked:
            assert np.array_equal(b.get(i), want[i]), (step, asked, i)
    b.free()
    for g in graphs:
        g.free()
