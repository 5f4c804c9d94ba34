"""Wait budgets that run out inside a team phase: one workgroup alone, a team of
two and the largest one stop at whichever iteration the budget ends in, every kernel
exits normally, the call returns INDIGO_ERR_TIMEOUT, and the same context then gives
exact results."""
import numpy as np
import pytest

from graphs import weighted

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("workgroups", [1, 9, 17, 0])
def test_budget_ends_inside_a_team_phase(ig, orc, ctx, workgroups):
    # 2^17 levels of two entries (one workgroup's, over 100 ms), and a mesh whose levels grow to a team's
    n = 1 << 17
    s = np.arange(n - 1)
    line = ig.from_edges(n, s.astype(np.int32), (s + 1).astype(np.int32), wseed=3, wmin=1, wmax=9)
    mesh = weighted(ig, ig.grid(1024, 1024), seed=2, wmax=100)
    dline, dmesh = ig.DeviceGraph(line), ig.DeviceGraph(mesh)
    ctx.set_hint(ig._lib.HINT_MAX_WORKGROUPS, workgroups)
    try:
        for budget in (1, 2, 3):
            ctx.set_hint(ig._lib.HINT_BUDGET_MS, budget)
            for name, dg in (("line", dline), ("mesh", dmesh)):
                for alg in (ctx.bfs, ctx.sssp):
                    print(f"budget {budget} ms, {workgroups} workgroups: {alg.__name__} {name}", flush=True)
                    with pytest.raises(ig.IndigoError) as e:
                        alg(dg, 0)
                    assert e.value.code == ig._lib.ERR_TIMEOUT
        ctx.set_hint(ig._lib.HINT_BUDGET_MS, 0)
        small = weighted(ig, ig.grid(40, 30), seed=5, wmax=9)
        dsmall = ig.DeviceGraph(small)
        assert np.array_equal(ctx.bfs(dsmall, 0), orc.bfs(small, 0))
        assert np.array_equal(ctx.sssp(dsmall, 0), orc.sssp(small, 0))
    finally:
        ctx.set_hint(ig._lib.HINT_BUDGET_MS, 0)
        ctx.set_hint(ig._lib.HINT_MAX_WORKGROUPS, 0)
