"""PageRank lists of more than 32 items of 1024 entries, whose finished items are
counted by groups of 32: around whole groups, with two and many of them, several such
vertices beside lists of few items, on grids with fewer waves than items and with more."""
import numpy as np
import pytest

from test_gpu_kernels import _pr_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workgroups", [1, 7, 0])
def test_items_counted_by_groups(ig, orc, ctx, workgroups):
    kib = 1024
    sizes = np.array([32 * kib - 2, 32 * kib - 1, 5000, 33 * kib - 2, 64 * kib - 2, 64 * kib - 1, 65 * kib - 2,
                      4096, 300 * kib + 17])
    k = len(sizes)
    n = k + 320 * kib
    rng = np.random.default_rng(9)
    src = np.concatenate([np.arange(k), np.repeat(np.arange(k), sizes), np.arange(k, n - 1)])
    dst = np.concatenate([(np.arange(k) + 1) % k] + [rng.permutation(n - k)[:s] + k for s in sizes]
                         + [np.arange(k + 1, n)])
    g = ig.from_edges(n, src.astype(np.int32), dst.astype(np.int32))
    items = -(-np.sort(g.degree)[::-1][:k] // kib)
    assert (items > 32).sum() >= 5 and (items <= 32).sum() >= 2
    dg = ig.DeviceGraph(g)
    ctx.set_hint(ig._lib.HINT_MAX_WORKGROUPS, workgroups)
    try:
        first, iters = ctx.pagerank(dg)
        again, iters2 = ctx.pagerank(dg)
    finally:
        ctx.set_hint(ig._lib.HINT_MAX_WORKGROUPS, 0)
    _pr_check(ig, orc, g, first, iters)
    assert iters2 == iters and np.array_equal(first, again)
