"""Batches whose scratch does not fit the free memory: an SSSP of many sources takes
them in several passes, a batch that does not fit even so is run in parts, and the
serving loop goes on with what it gets.  Results equal those of the single-query
kernels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _Filled:
    """All device memory taken but about `left` bytes."""

    def __init__(self, ig, left):
        self.ig, self.left, self.held = ig, left, []

    def __enter__(self):
        spare = self.ig.DeviceBuffer(self.left)
        size = 32 << 30
        while size >= 64 << 20:
            try:
                self.held.append(self.ig.DeviceBuffer(size))
            except self.ig.IndigoError:
                size //= 2
        spare.close()
        return self

    def __exit__(self, *exc):
        for b in self.held:
            b.close()


def test_batches_and_serving_in_little_memory(ig):
    """2^20 vertices and 1.2 GB: a query's scratch is 20 MB for one source a pass and 148
    for 32 (21 are rounded up to 32, 3 to 4), 90 queries do not fit at 20 each, and four
    serving slots' workspaces of two tasks of 32 sources do not fit beside the outputs."""
    g = ig.rmat(20, 4, seed=1, wmin=1, wmax=255)
    with ig.Context(0) as ctx:
        dg = ig.DeviceGraph(g)
        rng = np.random.default_rng(3)
        batches = []
        for queries, sources in ((12, 32), (20, 21), (40, 3), (90, 1)):
            qs = [ig.Query("sssp", 0, dg, rng.integers(0, g.nodes, sources)) for _ in range(queries)]
            for q in qs:
                q.out = ig.DeviceBuffer(4 * sources * g.nodes)
            batches.append(qs)
        n = 64
        src = rng.integers(0, g.nodes, n)
        outs = [ig.DeviceBuffer(4 * g.nodes) for _ in range(n)]
        with _Filled(ig, 1200 << 20):
            for qs in batches:
                print(f"{len(qs)} queries of {len(qs[0].sources)} sources", flush=True)
                ctx.batch([dg], qs)
                ctx.trim()
            print(f"serving {n} requests", flush=True)
            ig.serve([dg], ["sssp"] * n, np.zeros(n, np.int64), src, np.zeros(n), outs, slots=4, max_batch=64,
                     mem_budget=100 << 20)
        for qs in batches:
            for q in qs[:: len(qs) // 4]:
                got = q.result().reshape(len(q.sources), -1)
                for i in {0, len(q.sources) // 2, len(q.sources) - 1}:
                    assert np.array_equal(got[i], ctx.sssp(dg, int(q.sources[i]))), (len(qs), len(q.sources), i)
        for i in range(0, n, 9):
            assert np.array_equal(outs[i].to_array(np.int32, g.nodes), ctx.sssp(dg, int(src[i]))), i
        dg.close()
