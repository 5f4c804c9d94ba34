"""BFS, MIS and PageRank on graphs of many more vertices than entries (and of no
entries), whose passes over all vertices are the work."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes, links", [(1 << 20, 0), (1 << 20, 1), (1000003, 30000), (1 << 22, 3000)])
def test_many_vertices_few_entries(ig, orc, ctx, nodes, links):
    from test_gpu_kernels import _pr_check

    rng = np.random.default_rng(links)
    g = ig.from_edges(nodes, rng.integers(0, nodes, links).astype(np.int32), rng.integers(0, nodes, links).astype(np.int32))
    dg = ig.DeviceGraph(g)
    src = int(np.argmax(g.degree))
    assert np.array_equal(ctx.bfs(dg, src), orc.bfs(g, src))
    for signed in (False, True):
        assert np.array_equal(ctx.mis(dg, signed), orc.mis(g, signed))
    scores, iters = ctx.pagerank(dg)
    _pr_check(ig, orc, g, scores, iters)
