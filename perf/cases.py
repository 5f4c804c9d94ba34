"""Timed cases of the graph kernels' public entry points.

A case names an algorithm, a graph family with its sizes, and the option it
runs with; the graph's edges, its weights and the query's source come from a
seed.  Graphs are drawn with torch on the GPU, in the families that the
framework's own generators make (R-MAT a/b/c .57/.19/.19, Erdos-Renyi,
4-neighbour grids and road-like grids), and uploaded as a user's program
uploads its own: HostGraph, then DeviceGraph.  Results stay in device memory.

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  resident graph(s), source(s), result buffers, context
    run(state)           one call; returns its results
    exact(case, seed)    PageRank in float64 (the other results are integers)
    work(case)           bytes and operations that a pass cannot do without
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "parallelization-artifact-sc23_amd"))
import indigo2 as ig  # noqa: E402

BFS_SOURCES, SSSP_SOURCES = 64, 16  # per graph of a batch, as the batched benchmark has them
BATCH_ALGS = ("bfs", "sssp", "cc", "mis", "pr")


def listed():
    return [
        # the smallest call a user makes: one query on a small graph, where
        # launches, barriers and host calls are the time
        {"name": "bfs_rmat12", "alg": "bfs", "graph": "rmat", "scale": 12, "ef": 16},
        # the headline graph (R-MAT 22, edge factor 16), one call per algorithm
        {"name": "bfs_rmat22", "alg": "bfs", "graph": "rmat", "scale": 22, "ef": 16},
        {"name": "sssp_rmat22", "alg": "sssp", "graph": "rmat", "scale": 22, "ef": 16},
        {"name": "mis_rmat22", "alg": "mis", "graph": "rmat", "scale": 22, "ef": 16, "signed": False},
        {"name": "pr_rmat22", "alg": "pr", "graph": "rmat", "scale": 22, "ef": 16},
        {"name": "tc_rmat22", "alg": "tc", "graph": "rmat", "scale": 22, "ef": 16},
        # a social graph of ordinary size, as the serving pool holds many
        {"name": "sssp_rmat16", "alg": "sssp", "graph": "rmat", "scale": 16, "ef": 16},
        # high-diameter graphs: maps and meshes, thousands of narrow levels
        {"name": "bfs_grid1024", "alg": "bfs", "graph": "grid", "rows": 1024, "cols": 1024},
        {"name": "sssp_road1024", "alg": "sssp", "graph": "road", "rows": 1024, "cols": 1024},
        {"name": "cc_road2048", "alg": "cc", "graph": "road", "rows": 2048, "cols": 2048},
        # even degrees and a vertex count that no tile divides
        {"name": "pr_er1m", "alg": "pr", "graph": "er", "nodes": 1000003, "degree": 16},
        # many graphs of uneven sizes, many sources each, in one call
        {"name": "batch24", "alg": "batch", "graph": "mix", "count": 24, "lo": 1024, "hi": 131072},
    ]


def draw(rng):
    """A case of the listed ranges: every algorithm on the families it is run
    on, sizes log-uniform up to the listed ones' (deep graphs up to half of
    them, since a drawn shape may be up to four times as long as wide).  The
    full grid has no chance in it, so only the queries with a source or
    weights run there; triangles are counted on graphs that have some."""
    alg = rng.choice(["bfs", "sssp", "cc", "mis", "pr", "tc", "bfs", "sssp", "batch"])
    if alg == "batch":
        return {"alg": alg, "graph": "mix", "count": rng.randint(2, 24), "lo": 1024,
                "hi": int(2.0 ** rng.uniform(12, 17))}
    kind = rng.choice(["rmat", "rmat", "er"] if alg == "tc" else ["rmat", "rmat", "er", "grid", "road"])
    if kind == "grid" and alg not in ("bfs", "sssp"):
        kind = "road"
    case = {"alg": alg, "graph": kind}
    if kind == "rmat":
        case.update(scale=rng.randint(10, 21), ef=rng.randint(4, 16))
    elif kind == "er":
        case.update(nodes=int(2.0 ** rng.uniform(10, 21)) | 1,
                    degree=rng.randint(*{"cc": (2, 4), "tc": (12, 32)}.get(alg, (2, 32))))
    else:
        area, aspect = 2.0 ** rng.uniform(8, 19), 2.0 ** rng.uniform(-2, 2)
        rows = max(2, int(round(math.sqrt(area * aspect))))
        case.update(rows=rows, cols=max(2, int(area / rows)))
    if alg == "mis":
        case["signed"] = rng.random() < 0.5
    return case


# ---- graphs -------------------------------------------------------------------
def _rand(n, gen):
    return torch.rand(n, generator=gen, device="cuda")


def _rmat_pairs(scale, ef, gen):
    m = ef << scale
    src = torch.zeros(m, dtype=torch.int64, device="cuda")
    dst = torch.zeros_like(src)
    for _ in range(scale):
        r = _rand(m, gen)
        src = src * 2 + (r >= 0.76)
        dst = dst * 2 + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    return 1 << scale, src, dst


def _er_pairs(nodes, degree, gen):
    m = nodes * degree // 2
    return (nodes, torch.randint(nodes, (m,), generator=gen, device="cuda"),
            torch.randint(nodes, (m,), generator=gen, device="cuda"))


def _mesh_pairs(rows, cols, road, gen):
    """4-neighbour grid, ids row by row; a road keeps 85% of the links and adds
    2% of the diagonals."""
    n = rows * cols
    v = torch.arange(n, device="cuda")
    right, down = v[v % cols < cols - 1], v[: n - cols]
    diag = down[down % cols < cols - 1]
    if road:
        right, down = (x[_rand(len(x), gen) < 0.85] for x in (right, down))
        diag = diag[_rand(len(diag), gen) < 0.02]
    else:
        diag = diag[:0]
    return n, torch.cat([right, down, diag]), torch.cat([right + 1, down + cols, diag + cols + 1])


def _csr(nodes, src, dst, weight_max, seed):
    """Symmetric CSR without self loops and duplicates, lists sorted; weights
    in [1, weight_max], the same in both directions (0: none)."""
    keep = src != dst
    src, dst = src[keep], dst[keep]
    key = torch.cat([src * nodes + dst, dst * nodes + src])
    key = torch.unique_consecutive(torch.sort(key)[0])
    src, dst = key // nodes, key % nodes
    nindex = torch.zeros(nodes + 1, dtype=torch.int64, device="cuda")
    nindex[1:] = torch.cumsum(torch.bincount(src, minlength=nodes), 0)
    weight = None
    if weight_max:
        x = torch.minimum(src, dst) * 0x9E3779B1 + torch.maximum(src, dst) * 0x85EBCA77 + seed % 65521 * 0x27D4EB2F
        x = (x ^ (x >> 29)) * 0x2545F4914F6CDD1D
        weight = (1 + ((x >> 33) & 0x3FFFFFFF) % weight_max).to(torch.int32)
    return nindex.to(torch.int32), dst.to(torch.int32), weight


def _graph(case, seed, weighted):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["graph"]
    if kind == "rmat":
        nodes, src, dst = _rmat_pairs(case["scale"], case["ef"], gen)
    elif kind == "er":
        nodes, src, dst = _er_pairs(case["nodes"], case["degree"], gen)
    else:
        nodes, src, dst = _mesh_pairs(case["rows"], case["cols"], kind == "road", gen)
    return _csr(nodes, src, dst, (1000 if kind == "road" else 255) if weighted else 0, seed)


def _mix(case, seed):
    """The batch's graphs: vertex counts spread evenly over the logarithm of
    [lo, hi], even ones R-MAT with edge factor 8, odd ones Erdos-Renyi of
    average degree 8."""
    for i in range(case["count"]):
        n = int(round(case["lo"] * (case["hi"] / case["lo"]) ** ((i + 0.5) / case["count"])))
        one = ({"graph": "rmat", "scale": int(round(math.log2(n))), "ef": 8} if i % 2 == 0 else
               {"graph": "er", "nodes": n, "degree": 8})
        yield _graph(one, seed * 1000 + i, True)


def _upload(nindex, nlist, weight):
    host = ig.HostGraph(len(nindex) - 1, len(nlist), nindex.cpu().numpy(), nlist.cpu().numpy(),
                        None if weight is None else weight.cpu().numpy())
    return ig.DeviceGraph(host)


# ---- calls ----------------------------------------------------------------------
class TensorBuffer:
    """A result buffer in a torch tensor, passed where the framework takes a
    DeviceBuffer."""

    def __init__(self, tensor):
        self.tensor, self.ptr, self.nbytes = tensor, tensor.data_ptr(), 4 * tensor.numel()


@functools.lru_cache(maxsize=None)
def _context():
    return ig.Context(0)  # one per program, with its workspace


def _words(n):
    return torch.full((n,), -1, dtype=torch.int32, device="cuda")


def prepare(case, seed):
    alg = case["alg"]
    if alg == "batch":
        return _prepare_batch(case, seed)
    nindex, nlist, weight = _graph(case, seed, alg == "sssp")
    n = len(nindex) - 1
    state = {"alg": alg, "ctx": _context(), "graph": _upload(nindex, nlist, weight)}
    if alg in ("bfs", "sssp"):  # from a vertex that has neighbours, where there is one
        some = torch.nonzero(nindex[1:] > nindex[:-1]).flatten()
        state["src"] = int(some[np.random.default_rng(seed).integers(len(some))]) if len(some) else 0
    if alg == "mis":
        state["signed"] = case["signed"]
    if alg != "tc":
        state["out"] = TensorBuffer(_words(n))
    torch.cuda.synchronize()
    return state


def _prepare_batch(case, seed):
    rng = np.random.default_rng(seed)
    graphs = [_upload(*g) for g in _mix(case, seed)]
    queries, ints, pr = [], [], []
    for i, g in enumerate(graphs):
        for alg in BATCH_ALGS:
            k = {"bfs": BFS_SOURCES, "sssp": SSSP_SOURCES}.get(alg, 0)
            q = ig.Query(alg, i, g, rng.integers(0, g.nodes, k))
            (pr if alg == "pr" else ints).append((q, g.nodes + 1 if alg == "pr" else g.nodes * max(k, 1)))
            queries.append(q)
    whole = _words(sum(n for _, n in ints))  # all integer results in one tensor
    for (q, _), part in zip(ints, torch.split(whole, [n for _, n in ints])):
        q.out = TensorBuffer(part)
    for q, n in pr:
        q.out = TensorBuffer(_words(n))
    torch.cuda.synchronize()
    return {"alg": "batch", "ctx": _context(), "graphs": graphs, "queries": queries, "ints": whole,
            "pr": [q.out.tensor for q, _ in pr]}


def run(state):
    alg, ctx = state["alg"], state["ctx"]
    if alg == "batch":
        ctx.batch(state["graphs"], state["queries"])
        return {"ints": state["ints"], "scores": [p[:-1].view(torch.float32) for p in state["pr"]],
                "sweeps": [p[-1] for p in state["pr"]]}
    g = state["graph"]
    if alg == "tc":
        return {"triangles": ctx.tc(g)}
    out = state["out"]
    if alg == "bfs":
        ctx.bfs_into(g, state["src"], out)
    elif alg == "sssp":
        ctx.sssp_into(g, state["src"], out)
    elif alg == "cc":
        ctx.cc_into(g, out)
    elif alg == "mis":
        ctx.mis_into(g, out, state["signed"])
    else:
        sweeps = ctx.pagerank_into(g, out)
        return {"scores": out.tensor.view(torch.float32), "sweeps": sweeps}
    return {"out": out.tensor}


# ---- float64 PageRank and the work of a pass --------------------------------------
def _pagerank64(nindex, nlist):
    n = len(nindex) - 1
    deg = (nindex[1:] - nindex[:-1]).to(torch.int64)
    nlist = nlist.to(torch.int64)
    damp, eps = float(np.float32(0.85)), float(np.float32(1e-4))
    s = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    for _ in range(100):
        t = torch.segment_reduce((s / deg)[nlist], "sum", lengths=deg, initial=0, unsafe=True)
        new = (1.0 - damp) / n + damp * t
        change = float((new - s).abs().sum())
        s = new
        if not change > eps:
            break
    return s


def exact(case, seed):
    if case["alg"] == "pr":
        nindex, nlist, _ = _graph(case, seed, False)
        return {"scores": _pagerank64(nindex, nlist), "sweeps": None}
    if case["alg"] == "batch":
        return {"ints": None, "scores": [_pagerank64(g[0], g[1]) for g in _mix(case, seed)],
                "sweeps": [None] * case["count"]}
    return None


def _sizes(case):
    """(vertices, CSR entries), duplicates left in."""
    if case["graph"] == "rmat":
        return 1 << case["scale"], 2 * case["ef"] << case["scale"]
    if case["graph"] == "er":
        return case["nodes"], case["nodes"] * case["degree"]
    n = case["rows"] * case["cols"]
    return n, int(n * (3.44 if case["graph"] == "road" else 4.0))


def work(case):
    """The lists read once (with the weights where they are used) and the
    results written once; PageRank's additions of one sweep."""
    alg = case["alg"]
    if alg == "batch":
        n = case["count"] * (case["hi"] - case["lo"]) / math.log(case["hi"] / case["lo"])
        e = 12.0 * n
        return {"bytes": 5 * 4 * (n + e) + 4 * e + 4 * n * (BFS_SOURCES + SSSP_SOURCES + 3), "flops": e}
    n, e = _sizes(case)
    return {"bytes": 4.0 * (n + e + (e if alg == "sssp" else 0) + (0 if alg == "tc" else n)),
            "flops": float(e) if alg == "pr" else 0.0}
