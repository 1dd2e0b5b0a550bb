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
