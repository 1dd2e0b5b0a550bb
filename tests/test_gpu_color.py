"""np_color (GRAPH_COLOR_GPU) against the oracle: both methods bit-exact (int32 colors)."""
import os
import subprocess

import numpy as np
import pytest

from conftest import GOLDEN, PKG_DIR, free_bytes, load_golden, memory_is_back, random_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["rmat", "rmat_plain", "er", "grid", "multigraph", "tiny"])
def test_color_both_methods_match_oracle(npa, ctx, orc, kind):
    if kind == "rmat":
        G = npa.Graph.rmat(ctx, 13, 16, wmin=1, wmax=1, seed=61)
    elif kind == "rmat_plain":                       # ids not permuted: hubs at small ids
        G = npa.Graph.rmat(ctx, 12, 16, wmin=1, wmax=1, seed=62, permute=False)
    elif kind == "er":
        G = npa.Graph.er(ctx, 3000, 30000, 1, 1, seed=63)
    elif kind == "grid":
        G = npa.Graph.grid(ctx, 40, 50, None, 1, 1, seed=64)
    elif kind == "multigraph":
        rng = np.random.default_rng(65)
        row, col, _ = random_csr(rng, 2000, 12000, 1, 1)
        col[::5] = col[::5] % 7                       # parallel edges into small ids
        G = npa.Graph.from_csr(ctx, row, col, np.ones(len(col), np.int32))
    else:
        G = npa.Graph.from_csr(ctx, np.array([0, 1], np.int32), np.array([0], np.int32), np.ones(1, np.int32))
    row, col, _ = G.download()
    ref = orc.color(row, col)
    for method in (0, 1):
        got, st = ctx.color(G, method)
        assert np.array_equal(got, ref), (kind, method)
        assert st.iterations >= int(ref.max())
    G.free()


def test_color_rejects_bad_method(npa, ctx):
    G = npa.Graph.rmat(ctx, 8, 4, wmin=1, wmax=1, seed=66)
    with pytest.raises(npa.NpError):
        ctx.color(G, 2)
    G.free()


@pytest.mark.parametrize("solution", ["7", "12"])
def test_gpu_graph_color_cli_matches_oracle(tmp_path, orc, solution):
    g = load_golden("d9_rand.npz")
    out = tmp_path / "colors.txt"
    r = subprocess.run([os.path.join(PKG_DIR, "gpu-graph-color"), "-f", "0", "-i", os.path.join(GOLDEN, str(g["path"])),
                        "-s", solution, "-o", str(out)], cwd=tmp_path, stdout=subprocess.PIPE, stderr=subprocess.PIPE,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert "Execution time:" in r.stderr
    ref = orc.color(g["row"], g["col"])
    assert out.read_text().splitlines() == ["Node %d: %d" % (i + 1, c) for i, c in enumerate(ref)]


def _long_rows(n, lens, seed):
    """n vertices of 3 edges each, except vertex n - 1 - k, which has lens[k] (most to smaller ids)."""
    rng = np.random.default_rng(seed)
    deg = np.full(n, 3, np.int64)
    deg[n - len(lens):] = lens[::-1]
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(deg)
    return row, rng.integers(0, n, int(row[-1])).astype(np.int32)


@pytest.mark.parametrize("case", ["rows_at_ticket_edge", "long_rows", "long_rows_linked", "path", "path_down",
                                  "one_block_minus", "one_block", "one_block_plus", "empty_rows", "one_hub"])
def test_color_ticket_boundaries_match_oracle(npa, ctx, orc, case):
    """Tickets hold at most 256 edges inside blocks of 64 vertices: rows just below, at and above
    that, rows of many chunks, chunks that depend on one another, and the longest chains."""
    if case == "rows_at_ticket_edge":
        row, col = _long_rows(300, [255, 256, 257, 1, 0, 256, 511, 512, 513], 71)
    elif case == "long_rows":
        row, col = _long_rows(20000, [70000, 16385, 16384, 5000, 257], 72)
    elif case == "long_rows_linked":                  # every long row reads the long rows before it
        row, col = _long_rows(3000, [900] * 200, 73)
        col[row[2800]:] = 2800 + col[row[2800]:] % 200
    elif case in ("path", "path_down"):               # a chain of n dependencies, or none
        n = 5000
        row = np.minimum(np.arange(n + 1), n - 1).astype(np.int32)
        col = np.arange(1, n, dtype=np.int32)
        if case == "path":
            row = np.maximum(np.arange(n + 1) - 1, 0).astype(np.int32)
            col = np.arange(n - 1, dtype=np.int32)
    elif case == "empty_rows":
        row, col = np.zeros(1001, np.int32), np.zeros(0, np.int32)
    elif case == "one_hub":                           # more chunks than one look at the parts covers
        row, col = _long_rows(500, [256 * 150 + 1], 74)
    else:
        n = {"one_block_minus": 63, "one_block": 64, "one_block_plus": 65}[case]
        row, col = _long_rows(n, [4], 75)
    G = npa.Graph.from_csr(ctx, row, col, np.ones(len(col), np.int32))
    ref = orc.color(row, col)
    for _ in range(2):
        got, st = ctx.color(G)
        assert np.array_equal(got, ref), case
        assert st.iterations == int(ref.max())
    G.free()


def test_color_gives_back_large_buffers(npa, orc):
    """84 million vertices: the call's buffers take more than the 1 GiB that a context keeps, so the
    memory is back afterwards; same colors."""
    ctx = npa.Context(0)                              # nothing kept from other calls
    n = 80 << 20
    rng = np.random.default_rng(76)
    src = np.sort(rng.integers(0, n, 4000))
    row = np.zeros(n + 1, np.int32)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    col = np.where(rng.random(4000) < 0.5, src[rng.integers(0, 4000, 4000)], rng.integers(0, n, 4000)).astype(np.int32)
    G = npa.Graph.from_csr(ctx, row, col, np.ones(len(col), np.int32))
    before = free_bytes(npa)
    got, _ = ctx.color(G)
    assert memory_is_back(npa, before)
    assert np.array_equal(got, orc.color(row, col))
    G.free()
    ctx.close()
