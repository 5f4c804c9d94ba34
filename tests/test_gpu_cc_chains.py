"""Connected components of long thin graphs, whose union-find trees start as chains:
paths, rings, meshes of 16 columns and rows, and a chain of cliques (the Afforest
order), against labels in closed form; the vertex and the edge form and a batch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(ig, ctx, g, want):
    dg = ig.DeviceGraph(g)
    for variant in (ig._lib.VARIANT_VERTEX, ig._lib.VARIANT_EDGE):
        ctx.set_hint(ig._lib.HINT_VARIANT, variant)
        try:
            assert np.array_equal(ctx.cc(dg), want), variant
        finally:
            ctx.set_hint(ig._lib.HINT_VARIANT, 0)
    q = ig.Query("cc", 0, dg)
    ctx.batch([dg], [q])
    assert np.array_equal(q.result(), want)
    dg.close()


@pytest.mark.parametrize("n, cut", [(64, 0), (65, 0), (129, 0), (4097, 1000), (1 << 16, 0), (1 << 20, 0), (1 << 20, 65537)])
def test_cc_paths(ig, ctx, n, cut):
    """cut: every cut-th link is missing (0: none)."""
    s = np.arange(n - 1)
    s = s[(s + 1) % cut != 0] if cut else s
    g = ig.from_edges(n, s.astype(np.int32), (s + 1).astype(np.int32))
    _check(ig, ctx, g, np.arange(n) // cut * cut if cut else np.zeros(n, np.int64))


def test_cc_ring(ig, ctx):
    n = 1 << 20
    s = np.arange(n)
    _check(ig, ctx, ig.from_edges(n, s.astype(np.int32), ((s + 1) % n).astype(np.int32)), np.zeros(n, np.int64))


@pytest.mark.parametrize("rows, cols", [(65536, 16), (16, 65536), (16384, 64)])
def test_cc_thin_meshes(ig, ctx, rows, cols):
    _check(ig, ctx, ig.grid(rows, cols), np.zeros(rows * cols, np.int64))


def test_cc_chain_of_cliques(ig, ctx):
    k, c = 20000, 12
    a, b = np.triu_indices(c, 1)
    first = np.arange(k)[:, None] * c
    link = np.arange(k - 1) * c + c - 1
    g = ig.from_edges(k * c, np.concatenate([(first + a).ravel(), link]).astype(np.int32),
                      np.concatenate([(first + b).ravel(), link + 1]).astype(np.int32))
    _check(ig, ctx, g, np.zeros(k * c, np.int64))
