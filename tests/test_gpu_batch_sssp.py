"""Multi-source SSSP tasks of the batched engine on graphs that take a block's pairs each of
its ways: few active sources per entry (paths, meshes), most of them (complete
bipartite graphs, stars), some (random and R-MAT graphs); with split lists and without,
duplicate sources, and source counts around the powers of two that the rows are
rounded to.  Every row equals the single-query kernel's."""
import numpy as np
import pytest

from graphs import star, weighted

pytestmark = pytest.mark.gpu


def _graphs(ig):
    a, b = 70, 90
    bip = ig.from_edges(a + b, np.repeat(np.arange(a), b).astype(np.int32), np.tile(np.arange(a, a + b), a).astype(np.int32),
                        wseed=2, wmin=1, wmax=50)
    s = np.arange(299)
    line = ig.from_edges(300, s.astype(np.int32), (s + 1).astype(np.int32), wseed=3, wmin=1, wmax=9)
    return [line, bip, weighted(ig, star(ig, 5000), seed=4), ig.grid(41, 37, seed=5, wmin=1, wmax=100),
            ig.erdos_renyi(3001, 12000, seed=6, wmin=1, wmax=255), ig.rmat(12, 16, seed=7, wmin=1, wmax=255),
            ig.erdos_renyi(301, 150, seed=8, wmin=1, wmax=9)]


@pytest.mark.parametrize("gang", [1, 3, 0])
@pytest.mark.parametrize("sources", [1, 2, 3, 4, 5, 8, 16, 17, 31, 32])
def test_batched_sssp_rows(ig, ctx, sources, gang):
    gs = _graphs(ig)
    dgs = [ig.DeviceGraph(g) for g in gs]
    rng = np.random.default_rng(sources)
    qs = []
    for i, g in enumerate(gs):
        src = rng.integers(0, g.nodes, sources)
        src[-1] = src[0]  # the same source twice
        qs.append(ig.Query("sssp", i, dgs[i], src, gang=gang))
    ctx.batch(dgs, qs)
    for q in qs:
        got = q.result()
        for i, s in enumerate(q.sources):
            assert np.array_equal(got[i], ctx.sssp(dgs[q.graph], s)), (gs[q.graph].name, i)
