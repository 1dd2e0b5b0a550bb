"""np_bc (betweenness centrality, BC_GPU solution 7) against the oracle.

The GPU accumulates path counts and dependencies in double (parallel atomics: the summation
order varies) and returns float32, as the reference's float *bc; the bar is
|gpu - oracle| <= 1e-5 * |oracle| + 1e-5."""
import numpy as np
import pytest

from conftest import free_bytes, memory_is_back, random_csr

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-5, 1e-5


def _graph(npa, ctx, row, col):
    return npa.Graph.from_csr(ctx, row, col, np.ones(len(col), np.int32))


@pytest.mark.parametrize("n", [40, 300])   # 300: depth 299, forward levels in many growing runs
def test_bc_directed_path_closed_form(npa, ctx, n):
    row = np.minimum(np.arange(n + 1), n - 1).astype(np.int32)
    col = np.arange(1, n, dtype=np.int32)
    G = _graph(npa, ctx, row, col)
    bc, st = ctx.bc(G)
    assert np.allclose(bc, [v * (n - 1 - v) for v in range(n)], rtol=RTOL, atol=ATOL)
    assert st.iterations > 0
    G.free()


@pytest.mark.parametrize("kind", ["rmat", "er", "grid", "multigraph"])
def test_bc_every_vertex_matches_oracle(npa, ctx, orc, kind):
    """All sources (32 per batch): R-MAT with hubs, ER, a grid, and a multigraph with parallel
    edges, self loops and isolated vertices."""
    if kind == "rmat":
        G = npa.Graph.rmat(ctx, 10, 16, wmin=1, wmax=1, seed=51)
    elif kind == "er":
        G = npa.Graph.er(ctx, 700, 5000, 1, 1, seed=52)
    elif kind == "grid":
        G = npa.Graph.grid(ctx, 24, 30, None, 1, 1, seed=53)
    else:
        rng = np.random.default_rng(54)
        row, col, _ = random_csr(rng, 500, 3000, 1, 1)
        col[::7] = col[::7] % 20              # many parallel edges into a few vertices
        G = _graph(npa, ctx, row, col)
    row, col, _ = G.download()
    bc, _ = ctx.bc(G)
    ref = orc.bc(row, col)
    assert np.allclose(bc, ref, rtol=RTOL, atol=ATOL), float(np.max(np.abs(bc - ref)))
    G.free()


def test_bc_source_subsets(npa, ctx, orc):
    """Batch sizes 1, 5 (rows of 8 slots), 32 and 33 (a second batch of one), duplicate sources,
    a degree-0 source."""
    G = npa.Graph.rmat(ctx, 12, 8, wmin=1, wmax=1, seed=55)
    row, col, _ = G.download()
    deg = np.diff(row)
    zero = int(np.flatnonzero(deg == 0)[0])
    picks = [int(s) for s in npa.pick_sources(row, 40, 55)]
    for srcs in (picks[:1], picks[:5], picks[:32], picks[:33], [picks[0], picks[0], picks[1]], [zero] + picks[:3]):
        bc, st = ctx.bc(G, srcs)
        ref = orc.bc(row, col, srcs)
        assert np.allclose(bc, ref, rtol=RTOL, atol=ATOL), (len(srcs), float(np.max(np.abs(bc - ref))))
    G.free()


def test_bc_rejects_bad_sources(npa, ctx):
    G = npa.Graph.rmat(ctx, 8, 4, wmin=1, wmax=1, seed=56)
    with pytest.raises(npa.NpError):
        ctx.bc(G, [0, G.n])
    with pytest.raises(npa.NpError):
        ctx.bc(G, [-1])
    G.free()


@pytest.mark.parametrize("nsrc", [1, 2, 17, 32, 33])
def test_bc_rows_at_chunk_edges(npa, ctx, orc, nsrc):
    """Rows of out-degree 0, 1 and one below, at and one above each power of two up to 256 (a
    chunk holds 256 items or 64 edges, whichever split is in use), plus rows of several hundred
    edges; the targets lie two levels deep and share successors, so sums cross chunks."""
    degs = sorted({d for k in range(9) for d in (2 ** k - 1, 2 ** k, 2 ** k + 1)} | {512, 700})
    n = 1200
    rng = np.random.default_rng(57 + nsrc)
    deg = np.ones(n, np.int64)
    hubs = rng.permutation(n)[:2 * len(degs)]
    deg[hubs] = degs + degs
    row = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    col = rng.integers(0, n, row[-1]).astype(np.int32)
    G = _graph(npa, ctx, row, col)
    srcs = [int(s) for s in rng.permutation(n)[:nsrc]]
    srcs[0] = int(hubs[-1])
    bc, _ = ctx.bc(G, srcs)
    ref = orc.bc(row, col, srcs)
    assert np.allclose(bc, ref, rtol=RTOL, atol=ATOL), float(np.max(np.abs(bc - ref)))
    G.free()


def test_bc_overflowed_path_count_stays_with_its_source(npa, ctx, orc):
    """1,024 diamonds in a row give v 2^1024 shortest paths from A, past float64, and one from B along a
    path of the same length; v's only successor is one step from A.  So v has no successor for A, its
    infinite count multiplies nothing, and every dependency is finite."""
    k = 1024
    a = 3 * np.arange(k + 1)                       # a[0] = A, a[k] = v; the diamond's sides follow each a
    v, w, b = int(a[k]), int(a[k]) + 1, int(a[k]) + 2
    side = [(a[:-1], a[:-1] + 1), (a[:-1], a[:-1] + 2), (a[:-1] + 1, a[1:]), (a[:-1] + 2, a[1:])]
    chain = np.concatenate([b + np.arange(2 * k), [v]])     # B and 2 k - 1 more, then v
    src = np.concatenate([s for s, _ in side] + [chain[:-1], [v, a[0]]])
    dst = np.concatenate([d for _, d in side] + [chain[1:], [w, w]])
    order = np.argsort(src, kind="stable")
    row = np.zeros(b + 2 * k + 1, np.int64)
    np.add.at(row, src + 1, 1)
    row, col = np.cumsum(row).astype(np.int32), dst[order].astype(np.int32)
    G = _graph(npa, ctx, row, col)
    ref = orc.bc(row, col, [0, b])
    assert np.isfinite(ref).all()
    bc, _ = ctx.bc(G, [0, b])
    assert np.allclose(bc, ref, rtol=RTOL, atol=ATOL)
    G.free()


def test_bc_buffers_larger_than_the_kept_workspace(npa, orc):
    """13.6 million vertices: the call's buffers take more than 1 GiB, so it allocates and frees them
    itself; same results, and the memory is back afterwards."""
    ctx = npa.Context(0)                       # nothing kept from other calls
    n = 13 << 20
    rng = np.random.default_rng(58)
    src = np.sort(rng.integers(0, 3000, 20000))
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    col = rng.integers(0, 3000, 20000).astype(np.int32)
    G = _graph(npa, ctx, row, col)
    before = free_bytes(npa)
    bc, _ = ctx.bc(G, [int(src[0])])
    assert memory_is_back(npa, before)
    ref = orc.bc(row, col, [int(src[0])])
    assert np.allclose(bc, ref, rtol=RTOL, atol=ATOL)
    G.free()
    ctx.close()
