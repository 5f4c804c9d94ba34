"""PageRank, call after call, on graphs of few long lists and many workgroups
without any of their items: sweep counts and scores are the same bit for bit."""
import numpy as np
import pytest

from test_gpu_kernels import _pr_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hubs,leaves", [(1, 1 << 14), (1, 1 << 18), (5, 30000)])
def test_repeated_calls_agree(ig, orc, ctx, hubs, leaves):
    src = np.concatenate([np.repeat(np.arange(hubs), leaves), np.arange(hubs - 1)])
    dst = np.concatenate([hubs + np.arange(hubs * leaves), np.arange(1, hubs)])
    g = ig.from_edges(hubs * (leaves + 1), src.astype(np.int32), dst.astype(np.int32))
    dg = ig.DeviceGraph(g)
    ctx.set_hint(ig._lib.HINT_BUDGET_MS, 3000)
    try:
        first, iters = ctx.pagerank(dg)
        _pr_check(ig, orc, g, first, iters)
        for _ in range(40):
            scores, n = ctx.pagerank(dg)
            assert n == iters and np.array_equal(scores, first)
    finally:
        ctx.set_hint(ig._lib.HINT_BUDGET_MS, 0)
