"""SSSP splits that move more parked vertices into the near frontier than a team's
shares hold (1024 each), and piles beyond what its members park (2048 each):
what does not fit goes to the grid, and the distances stay exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def layers(ig, width, depth, leaves):
    """A source, `depth` layers of `width` vertices joined by weight 1, and at each of
    their vertices `leaves` paths of two edges, of weights 5000 and 3."""
    n = width * depth
    v = 1 + np.arange(n)
    first = 1 + n + np.arange(n * leaves)
    second = first + n * leaves
    src = np.concatenate([np.zeros(width, int), v[:-width] if depth > 1 else v[:0], np.repeat(v, leaves), first])
    dst = np.concatenate([v[:width], v[width:], first, second])
    w = np.concatenate([np.ones(n, int), np.full(n * leaves, 5000), np.full(n * leaves, 3)])
    total = 1 + n + 2 * n * leaves
    order = np.lexsort((np.concatenate([dst, src]), np.concatenate([src, dst])))
    a = np.concatenate([src, dst])[order]
    index = np.concatenate([[0], np.cumsum(np.bincount(a, minlength=total))])
    return ig.HostGraph(total, len(a), index.astype(np.int32), np.concatenate([dst, src])[order].astype(np.int32),
                        np.concatenate([w, w])[order].astype(np.int32))


@pytest.mark.parametrize("width,depth,workgroups", [
    (512, 16, 0),    # the largest team, 65536 parked: one split fills every share
    (512, 24, 0),    # ... and more than its members park
    (512, 9, 0),     # about 32 shares
    (128, 5, 24),    # a team of three
    (128, 16, 24),
    (48, 4, 0),      # one workgroup: 1536 parked
    (48, 4, 8),
    (40, 8, 1),      # ... more than it parks
])
@pytest.mark.parametrize("delta", [100, 4000])
def test_split_overfills_the_shares(ig, orc, ctx, width, depth, workgroups, delta):
    g = layers(ig, width, depth, 8)
    dg = ig.DeviceGraph(g)
    want = orc.sssp(g, 0)
    ctx.set_hint(ig._lib.HINT_SSSP_DELTA, delta)
    ctx.set_hint(ig._lib.HINT_MAX_WORKGROUPS, workgroups)
    try:
        for call in range(4):
            print(f"{depth} layers of {width}, {workgroups} workgroups, delta {delta}, call {call}", flush=True)
            assert np.array_equal(ctx.sssp(dg, 0), want)
    finally:
        ctx.set_hint(ig._lib.HINT_SSSP_DELTA, 0)
        ctx.set_hint(ig._lib.HINT_MAX_WORKGROUPS, 0)
