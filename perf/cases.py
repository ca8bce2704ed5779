"""The graph workloads this framework is used for, as measurable cases.

Every case is one call (or the short sequence of calls that its command-line
tool makes) of a public entry point on graphs that live on the GPU: SSSP and
BFS from one source, direction-optimising BFS, many sources of one graph in
one launch, many graphs in one launch, connected components and PageRank.
Graphs are the three families of the benchmark configurations -- 4-neighbour
grids, road-like grids and RMAT -- made on the GPU with torch from the seed,
in the distributions of lsg_gen_grid, lsg_gen_roadlike and lsg_gen_rmat, and
handed to the library as torch tensors (DeviceGraph.wrap).
"""
from __future__ import annotations

import numpy as np
import torch

from galoisgpu_amd import Options
from galoisgpu_amd import sched as lsched
from galoisgpu_amd.apps import bfs_do_into, bfs_into, cc_into, pagerank_into, sssp_into
from galoisgpu_amd.batch import sssp_graphs, sssp_multi_into
from galoisgpu_amd.graph import DeviceGraph

INF = 0x7FFFFFFF
DEV = "cuda:0"


def listed():
    return [
        # The smallest call: the 64x64 grid of the smoke test; launch and round latency only.
        {"name": "sssp_grid_64", "op": "sssp", "family": "grid", "rows": 64, "cols": 64, "delta": 32},
        # Configuration 1: a 256x256 grid, about 1200 rounds of a few hundred vertices.
        {"name": "sssp_grid_256", "op": "sssp", "family": "grid", "rows": 256, "cols": 256, "delta": 32},
        # Configuration 2: RMAT-20 from its largest hub; few, wide rounds and skewed degrees.
        {"name": "sssp_rmat_20", "op": "sssp", "family": "rmat", "n": 1 << 20, "ef": 16, "delta": 32},
        # Configuration 3: a 2048x2048 road-like network, the reference's default delta.
        {"name": "sssp_road_2048", "op": "sssp", "family": "road", "rows": 2048, "cols": 2048, "delta": 10000},
        # Configuration 2's BFS: the plain level-synchronous app.
        {"name": "bfs_rmat_20", "op": "bfs", "family": "rmat", "n": 1 << 20, "ef": 16},
        # BFS on a road-like network of odd sides: many narrow levels.
        {"name": "bfs_road_1023x777", "op": "bfs", "family": "road", "rows": 1023, "cols": 777},
        # Direction-optimising BFS on a large graph whose reverse the program keeps.
        {"name": "bfs_do_rmat_22", "op": "bfs_do", "family": "rmat", "n": 1 << 22, "ef": 16},
        # A small batch of sources, ragged in every size, with the default options.
        {"name": "multi_rmat_100003_s9", "op": "multi", "family": "rmat", "n": 100003, "ef": 16, "nsrc": 9,
         "delta": 32, "sched": False},
        # The headline: 64 uniform sources of RMAT-22 in one launch, learned schedule, captured graph.
        {"name": "multi_rmat_22_s64", "op": "multi", "family": "rmat", "n": 1 << 22, "ef": 16, "nsrc": 64,
         "delta": 32, "sched": True},
        # Configuration 4B's mixture (scales 10 to 16, ef 8) as one batch of 64 graphs.
        {"name": "graphs_64", "op": "graphs", "family": "rmat", "count": 64, "lo": 10, "hi": 16, "ef": 8,
         "delta": 32},
        # Connected components of a large skewed graph (apps/cc).
        {"name": "cc_rmat_22", "op": "cc", "family": "rmat", "n": 1 << 22, "ef": 16},
        # PageRank as the pr tool runs it: reverse CSR, then the fixpoint (apps/pr).
        {"name": "pagerank_rmat_22", "op": "pagerank", "family": "rmat", "n": 1 << 22, "ef": 16},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    """One more case of the same ranges, sizes spread over their logarithm."""
    op = rng.choice(["sssp", "sssp", "bfs", "bfs_do", "multi", "multi", "graphs", "cc", "pagerank"])
    if op == "graphs":
        lo = rng.randint(8, 12)
        return {"op": op, "family": "rmat", "count": _log_uniform(rng, 5, 64), "lo": lo,
                "hi": rng.randint(lo + 1, 16), "ef": rng.choice([8, 16]), "delta": rng.choice([32, 100, 1000])}
    family = rng.choice({"sssp": ["grid", "road", "rmat"], "bfs": ["grid", "road", "rmat"], "bfs_do": ["rmat", "road"],
                         "multi": ["rmat"], "cc": ["road", "rmat"], "pagerank": ["road", "rmat"]}[op])
    c = {"op": op, "family": family}
    if family == "grid":
        c.update(rows=_log_uniform(rng, 40, 512), cols=_log_uniform(rng, 40, 512))
    elif family == "road":
        c.update(rows=_log_uniform(rng, 128, 2048), cols=_log_uniform(rng, 128, 2048))
    else:
        c.update(n=_log_uniform(rng, 1 << 14, 1 << 22), ef=rng.choice([8, 16]))
    if op == "sssp":
        c["delta"] = {"grid": rng.choice([32, 256]), "road": rng.choice([2000, 10000]),
                      "rmat": rng.choice([32, 128])}[family]
    if op == "multi":
        c["sched"] = rng.random() < 0.7
        if not c["sched"]:
            c["n"] = min(c["n"], (1 << 18) + rng.randint(1, 999))
        c.update(nsrc=rng.randint(2, 64), delta=32)
    return c


# ---- inputs -----------------------------------------------------------------


def _csr(n, src, dst, wlo, whi, gen):
    """Sorted CSR without self loops and duplicates, weights U[wlo, whi] per directed edge (int32 tensors)."""
    keep = src != dst
    key = torch.unique(src[keep] * n + dst[keep])
    src = torch.div(key, n, rounding_mode="floor")
    row = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    row[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0)
    w = torch.randint(wlo, whi + 1, (key.numel(),), generator=gen, device=DEV, dtype=torch.int32)
    return row.to(torch.int32), (key - src * n).to(torch.int32), w


def _rmat(n, ef, gen):
    """Directed RMAT (0.57, 0.19, 0.19); pairs with an end at n or above are dropped."""
    scale = max(1, (n - 1).bit_length())
    m = ef * n
    src = torch.zeros(m, dtype=torch.int64, device=DEV)
    dst = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(scale):
        r = torch.rand(m, generator=gen, device=DEV)
        src.mul_(2).add_(r >= 0.76)
        dst.mul_(2).add_(((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    if n < 1 << scale:
        keep = (src < n) & (dst < n)
        src, dst = src[keep], dst[keep]
    return _csr(n, src, dst, 1, 255, gen)


def _lattice(rows, cols, gen, drop):
    """Undirected edges (u, v) of a rows x cols grid, each but the first corner's kept with probability 1 - drop."""
    ids = torch.arange(rows * cols, device=DEV).view(rows, cols)
    u = torch.cat([ids[:, :-1].reshape(-1), ids[:-1].reshape(-1)])
    v = torch.cat([ids[:, 1:].reshape(-1), ids[1:].reshape(-1)])
    if drop:
        keep = (torch.rand(u.numel(), generator=gen, device=DEV) >= drop) | (u == 0)
        u, v = u[keep], v[keep]
    return u, v


def _graph(case, gen):
    if case["family"] == "rmat":
        return _rmat(case["n"], case["ef"], gen)
    n = case["rows"] * case["cols"]
    if case["family"] == "grid":
        u, v = _lattice(case["rows"], case["cols"], gen, 0.0)
        return _csr(n, torch.cat([u, v]), torch.cat([v, u]), 1, 100, gen)
    u, v = _lattice(case["rows"], case["cols"], gen, 0.10)
    extra = torch.randint(0, n, (2, int(round(0.001 * u.numel()))), generator=gen, device=DEV)
    u, v = torch.cat([u, extra[0]]), torch.cat([v, extra[1]])
    return _csr(n, torch.cat([u, v]), torch.cat([v, u]), 1, 10000, gen)


def _inputs(case, seed):
    """The graphs (row, dst, weight) of a case and its sources."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed))
    if case["op"] == "graphs":
        # sizes between powers of two as well, the same for every seed; one graph of each end of the range is always there
        rng = np.random.default_rng(case["count"])
        sizes = [1 << case["lo"], 1 << case["hi"]] + [
            int(round(2.0 ** rng.uniform(case["lo"], case["hi"]))) for _ in range(case["count"] - 2)]
        graphs = [_rmat(n, case["ef"], gen) for n in sizes]
        return graphs, [int(torch.argmax(g[0].diff())) for g in graphs]
    g = _graph(case, gen)
    n = g[0].numel() - 1
    if case["op"] == "multi":
        return [g], [int(x) for x in np.random.default_rng(int(seed)).integers(0, n, case["nsrc"])]
    return [g], [int(torch.argmax(g[0].diff())) if case["family"] == "rmat" else 0]


class _Matrix:
    """A torch tensor as the [V][S] result matrix of sssp_multi_into."""

    def __init__(self, t):
        self.ptr, self.nbytes = t.data_ptr(), t.numel() * t.element_size()


def _wrap(g):
    row, dst, w = g
    return DeviceGraph.wrap(row.numel() - 1, dst.numel(), row.data_ptr(), dst.data_ptr(), w.data_ptr())


def prepare(case, seed):
    graphs, srcs = _inputs(case, seed)
    torch.cuda.synchronize()  # the library runs on its own stream
    s = {"op": case["op"], "tensors": graphs, "devs": [_wrap(g) for g in graphs], "srcs": srcs}
    dev = s["devs"][0]
    if case["op"] == "multi":
        s["out"] = torch.empty((dev.nnodes, len(srcs)), dtype=torch.int32, device=DEV)
        s["matrix"] = _Matrix(s["out"])
        s["opts"] = Options(delta=case["delta"])
        if case["sched"]:
            lsched.load_model(lsched.default_model_path("batched"), kind="batched")
            s["opts"] = Options(delta=case["delta"], block_size=256, heavy_deg=256, sched=1, graph_launch=True)
    elif case["op"] == "graphs":
        s["opts"] = Options(delta=case["delta"])
    else:
        s["out"] = torch.empty(dev.nnodes, dtype=torch.float32 if case["op"] == "pagerank" else torch.int32, device=DEV)
        if case["op"] in ("sssp", "bfs"):
            s["opts"] = Options(delta=case.get("delta", 10000), start_node=srcs[0])
        if case["op"] == "bfs_do":
            s["rev"] = dev.transpose()
    return s


def run(s):
    op, dev = s["op"], s["devs"][0]
    if op == "graphs":
        return sssp_graphs(s["devs"], s["srcs"], s["opts"])[0]
    if op == "multi":
        sssp_multi_into(dev, s["srcs"], s["opts"], s["matrix"])
    elif op == "sssp":
        sssp_into(dev, s["out"].data_ptr(), s["opts"])
    elif op == "bfs":
        bfs_into(dev, s["out"].data_ptr(), s["opts"])
    elif op == "bfs_do":
        bfs_do_into(dev, s["rev"], s["out"].data_ptr(), s["srcs"][0])
    elif op == "cc":
        cc_into(dev, s["out"].data_ptr())
    else:
        rev = dev.transpose()
        pagerank_into(dev, rev, s["out"].data_ptr())
        rev.close()
    return s["out"]


def work(case):
    """Bytes of the graph read once and the result written once; one operation per edge and source."""
    if case["op"] == "graphs":
        lo, hi = case["lo"], case["hi"]
        n = int(case["count"] * (2.0 ** hi - 2.0 ** lo) / ((hi - lo) * 0.6931))
        e = 0.9 * n * case["ef"]
    elif case["family"] == "rmat":
        n = case["n"]
        e = 0.95 * n * case["ef"]
    else:
        n = case["rows"] * case["cols"]
        e = 4.0 * n if case["family"] == "grid" else 3.6 * n
    per_edge = 8 if case["op"] in ("sssp", "multi", "graphs") else 4
    nsrc = case.get("nsrc", 1)
    return {"bytes": per_edge * e + 4.0 * n + 4.0 * n * nsrc, "flops": e * nsrc}


# ---- results in 64 bits -------------------------------------------------------


def _edges(g):
    row, dst, w = (t.to(torch.int64) for t in g)
    src = torch.repeat_interleave(torch.arange(row.numel() - 1, device=DEV), row.diff())
    return src, dst, w, row.diff()


def _distances(g, source, unit):
    """Bellman-Ford in int64; unit: every edge has length 1."""
    src, dst, w, _ = _edges(g)
    w = torch.ones_like(w) if unit else w
    d = torch.full((g[0].numel() - 1,), INF, dtype=torch.int64, device=DEV)
    d[source] = 0
    while True:
        new = d.scatter_reduce(0, dst, d[src] + w, "amin")
        if torch.equal(new, d):
            return d.to(torch.int32)
        d = new


def _components(g):
    """Smallest vertex id of each vertex's component: label propagation with pointer jumping."""
    src, dst, _, _ = _edges(g)
    label = torch.arange(g[0].numel() - 1, device=DEV)
    while True:
        new = label.scatter_reduce(0, dst, label[src], "amin").scatter_reduce(0, src, label[dst], "amin")
        new = torch.minimum(new, new[new])
        new = new[new]
        if torch.equal(new, label):
            return label.to(torch.int32)
        label = new


def _ranks(g):
    """PageRank's fixpoint (damping 0.85) in float64; in-edges summed as differences of one running sum."""
    src, dst, _, deg = _edges(g)
    n = deg.numel()
    order = torch.argsort(dst)
    src = src[order]
    ends = torch.cumsum(torch.bincount(dst, minlength=n), 0)
    share = 0.85 / deg.clamp(min=1).to(torch.float64)
    p = torch.full((n,), 0.15, dtype=torch.float64, device=DEV)
    total = torch.zeros(src.numel() + 1, dtype=torch.float64, device=DEV)
    for _ in range(200):
        torch.cumsum((p * share)[src], 0, out=total[1:])
        new = 0.15 + torch.diff(total[ends], prepend=total[:1])
        moved = float(((new - p).abs() / new).max())
        p = new
        if moved < 1e-11:
            break
    return p


def exact(case, seed):
    if case["op"] in ("multi", "graphs"):
        return None  # whole numbers of one traversal per source; the single-source cases cover them
    if case["family"] != "rmat" and case["op"] in ("sssp", "bfs"):
        return None  # thousands of rounds over all edges
    (g,), (source,) = _inputs(case, seed)
    if case["op"] == "pagerank":
        return _ranks(g)
    if case["op"] == "cc":
        return _components(g)
    return _distances(g, source, case["op"] != "sssp")
