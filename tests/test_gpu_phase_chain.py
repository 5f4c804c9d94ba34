"""BFS and SSSP on graphs whose team phases follow each other without a pass of the
whole grid in between, are entered with an empty near frontier, and run several
splits: what one phase leaves, and the piles that it clears, are read by
workgroups that may be late.  Exact results, call after call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def clique_chain(ig, k, c, wmax):
    a, b = np.triu_indices(c, 1)
    base = np.arange(k)[:, None] * c
    link = np.arange(k - 1) * c + c - 1
    src = np.concatenate([(base + a).ravel(), link])
    dst = np.concatenate([(base + b).ravel(), link + 1])
    return ig.from_edges(k * c, src.astype(np.int32), dst.astype(np.int32), wseed=4, wmin=1, wmax=wmax)


def star_chain(ig, k, leaves):
    """Hubs in a row, each with leaves: levels of one workgroup and of a team in turn."""
    hub = np.arange(k) * (leaves + 1)
    leaf = hub[:, None] + 1 + np.arange(leaves)
    src = np.concatenate([np.repeat(hub, leaves), hub[:-1]])
    dst = np.concatenate([leaf.ravel(), hub[1:]])
    return ig.from_edges(k * (leaves + 1), src.astype(np.int32), dst.astype(np.int32), wseed=5, wmin=1, wmax=1000)


@pytest.mark.parametrize("name", ["cliques 64x100", "cliques 256x40", "cliques 64x12", "stars 64x700", "stars 40x3000"])
@pytest.mark.parametrize("delta", [0, 40])
def test_consecutive_phases(ig, orc, ctx, name, delta):
    kind, size = name.split()
    k, c = (int(x) for x in size.split("x"))
    g = clique_chain(ig, k, c, 255) if kind == "cliques" else star_chain(ig, k, c)
    dg = ig.DeviceGraph(g)
    ctx.set_hint(ig._lib.HINT_BUDGET_MS, 3000)
    ctx.set_hint(ig._lib.HINT_SSSP_DELTA, delta)
    try:
        for src in (0, g.nodes - 1, g.nodes // 2):
            want = orc.sssp(g, src)
            levels = orc.bfs(g, src)
            for call in range(8):
                print(f"{name}, delta {delta}, source {src}, call {call}", flush=True)
                assert np.array_equal(ctx.sssp(dg, src), want)
                assert np.array_equal(ctx.bfs(dg, src), levels)
    finally:
        ctx.set_hint(ig._lib.HINT_BUDGET_MS, 0)
        ctx.set_hint(ig._lib.HINT_SSSP_DELTA, 0)
