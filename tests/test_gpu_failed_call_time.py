"""The device time that a context reports after a call that failed is that call's
own: one that ran out of its wait budget took at least the budget, and one that was
refused on the device did not take as long as the call before it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_time_of_a_call_that_failed(ig, ctx):
    n = 1 << 17
    s = np.arange(n - 1)
    line = ig.from_edges(n, s.astype(np.int32), (s + 1).astype(np.int32), wseed=3, wmin=1, wmax=9)
    tiny = ig.grid(8, 8, seed=1, wmin=1, wmax=9)
    dline, dtiny = ig.DeviceGraph(line), ig.DeviceGraph(tiny)
    for alg in (ctx.bfs, ctx.sssp):
        alg(dtiny, 0)
        assert ctx.last_ms < 3.0
        ctx.set_hint(ig._lib.HINT_BUDGET_MS, 4)
        try:
            with pytest.raises(ig.IndigoError) as e:
                alg(dline, 0)
        finally:
            ctx.set_hint(ig._lib.HINT_BUDGET_MS, 0)
        assert e.value.code == ig._lib.ERR_TIMEOUT
        assert ctx.last_ms >= 4.0
        assert ctx.last_kernel[1] >= 4.0
    v = int(np.flatnonzero(tiny.degree >= 2)[0])
    b = tiny.nindex[v]
    nl = tiny.nlist.copy()
    nl[b], nl[b + 1] = nl[b + 1], nl[b]
    unsorted = ig.DeviceGraph(ig.HostGraph(tiny.nodes, tiny.edges, tiny.nindex, nl))
    mesh = ig.DeviceGraph(ig.grid(1024, 1024))
    ctx.bfs(mesh, 0)
    before = ctx.last_ms
    with pytest.raises(ig.IndigoError) as e:
        ctx.tc(unsorted)
    assert e.value.code == ig._lib.ERR_UNSORTED
    assert ctx.last_ms < before
    assert ctx.last_kernel[0] != "bfs_kernel"
