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


@pytest.mark.parametrize("gang", [2, 5, 64, 0])
def test_narrow_levels_of_a_gang(ig, ctx, gang):
    """Levels of a few entries, which member 0 runs alone, before, between and after
    wide ones: a line through a random graph's vertices, a chain of cliques, stars on
    a line and a line alone."""
    n, k = 4000, 30
    s = np.arange(n - 1)
    rnd = np.random.default_rng(1)
    line = (s, s + 1)
    wide = (np.concatenate([s, rnd.integers(1500, 2500, 9000)]), np.concatenate([s + 1, rnd.integers(1500, 2500, 9000)]))
    a, b = np.triu_indices(12, 1)
    first = np.arange(200)[:, None] * 12
    link = np.arange(199) * 12 + 11
    cliques = (np.concatenate([(first + a).ravel(), link]), np.concatenate([(first + b).ravel(), link + 1]))
    p = np.arange(k - 1) * 700
    stars = (np.concatenate([p, np.repeat(np.arange(k) * 700, 699)]),
             np.concatenate([p + 700, np.delete(np.arange(k * 700), np.arange(k) * 700)]))
    gs = [ig.from_edges(int(max(x.max(), y.max())) + 1, x.astype(np.int32), y.astype(np.int32), wseed=5, wmin=1, wmax=60)
          for x, y in (line, wide, cliques, stars)]
    dgs = [ig.DeviceGraph(g) for g in gs]
    qs = []
    for i, g in enumerate(gs):
        for alg, count in (("bfs", 1), ("bfs", 5), ("bfs", 64), ("sssp", 1), ("sssp", 3), ("sssp", 16)):
            qs.append(ig.Query(alg, i, dgs[i], rnd.integers(0, g.nodes, count), gang=gang))
    ctx.batch(dgs, qs)
    for q in qs:
        got = q.result()
        alone = ctx.bfs if q.name == "bfs" else ctx.sssp
        for i in range(0, len(q.sources), max(1, len(q.sources) // 5)):
            assert np.array_equal(got[i], alone(dgs[q.graph], q.sources[i])), (q.graph, q.name, i)
