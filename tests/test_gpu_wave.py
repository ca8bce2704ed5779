"""The wavefront traversal kernel (default options of sssp/bfs) at the edges of
its units, piles and modes, against the host oracle.  Distances are whole
numbers: equality."""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph, Options
from galoisgpu_amd.apps import bfs_gg_main, sssp_gg_main

pytestmark = pytest.mark.gpu


def csr(n, edges):
    """CSRGraph of (src, dst, weight) rows."""
    e = np.asarray(edges, dtype=np.int64).reshape(-1, 3)
    e = e[np.argsort(e[:, 0], kind="stable")]
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(e[:, 0], minlength=n))
    return CSRGraph.from_arrays(row, e[:, 1], e[:, 2])


def tree(*degrees):
    """Every vertex of depth k has degrees[k] children; some cross edges."""
    edges, level, n = [], [0], 1
    rng = np.random.default_rng(sum(degrees))
    for d in degrees:
        nxt = []
        for u in level:
            for _ in range(d):
                edges.append((u, n, int(rng.integers(1, 100))))
                nxt.append(n)
                n += 1
        level = nxt
    for _ in range(n // 2):
        edges.append((int(rng.integers(n)), int(rng.integers(n)), int(rng.integers(1, 100))))
    return csr(n, edges)


def check(g, src, delta, **kw):
    dev = g.copy_to_gpu()
    print("wave", g.nnodes, g.nedges, src, delta, kw, flush=True)
    sssp_gg_main(g, dev, Options(delta=delta, start_node=src, **kw))
    dev.copy_to_cpu(g)
    assert np.array_equal(g.node_data, oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, src))
    bfs_gg_main(g, dev, Options(start_node=src, **kw))
    dev.copy_to_cpu(g)
    assert np.array_equal(g.node_data, oracle.bfs(g.row_start, g.edge_dst, src)[0])
    dev.close()


# Heavy threshold (256 edges by default), rounds of one block (512 items), its
# piles (1024 entries), staged items (256 a wavefront) and heavy items (32).
@pytest.mark.parametrize("degrees", [(1,), (255,), (256, 1, 1), (257,), (8, 64), (8, 64, 1, 1), (19, 27, 2), (4, 255, 1),
                                     (4, 256, 1), (200, 6), (3, 2, 300), (40, 260, 1)])
def test_trees(degrees):
    g = tree(*degrees)
    for delta in (1, 40, 10000):
        check(g, 0, delta, block_size=256)
        check(g, 0, delta)  # up to 32768 vertices: the one-workgroup kernel


@pytest.mark.parametrize("kw", [dict(block_size=b, grid_blocks=n) for b in (256, 512, 1024) for n in (1, 7, 16, 17, 300)]
                         + [dict(heavy_deg=300), dict(heavy_deg=2**31 - 1), dict(graph_launch=True)])
def test_launch_shapes(kw):
    g = CSRGraph.rmat(13, 8, seed=3)
    check(g, g.max_degree_vertex(), 32, **kw)
    check(CSRGraph.grid(37, 53, seed=2), 5, 64, **kw)


# Low-degree graphs, whose threshold moves in growing steps: up to one that passes every distance.
@pytest.mark.parametrize("rows,cols,whi", [(1, 3000, 9), (64, 64, 100), (90, 131, 1 << 20), (300, 410, 60000)])
def test_paced_threshold(rows, cols, whi):
    g = CSRGraph.grid(rows, cols, 1, whi, seed=rows)
    for delta in (1, 32, 5000, 1 << 30):
        check(g, 7, delta, block_size=256)
        check(g, 7, delta)


# Wavefronts that go on with what they pushed: levels are still reported one by one.
@pytest.mark.parametrize("rows,cols", [(182, 182), (700, 90), (3, 30000)])
def test_hops(rows, cols):
    g = CSRGraph.roadlike(rows, cols, 0.1, 0.001, 1, 1000, seed=rows)
    for delta in (20, 1000, 1 << 28):
        check(g, 11, delta)
    dev = g.copy_to_gpu()
    st = bfs_gg_main(g, dev, Options(start_node=11))
    dev.copy_to_cpu(g)
    reached = g.node_data[g.node_data != 2**31 - 1]
    assert st["iterations"] == st["near_iters"] == reached.max() + 1
    dev.close()


# The one-workgroup kernel: both sides of its largest size, rounds of more
# vertices than it lists (4096), heavy vertices (32 edges), the array's last edges.
@pytest.mark.parametrize("n,kind", [(32768, "grid"), (32769, "grid"), (32768, "star"), (32767, "star"), (30000, "random"),
                                    (5, "star"), (2, "star"), (1, "star")])
def test_one_workgroup(n, kind):
    rng = np.random.default_rng(n)
    if kind == "grid":
        g = CSRGraph.grid(128, n // 128, 1, 1000, seed=1) if n % 128 == 0 else CSRGraph.grid(3, n // 3, 1, 1000, seed=1)
    elif kind == "star":  # the hub's round pushes every other vertex at once
        v = np.arange(1, n)
        g = csr(n, np.stack([np.concatenate([v, np.zeros(n - 1, int)]), np.concatenate([np.zeros(n - 1, int), v]),
                             rng.integers(1, 50, 2 * (n - 1))], axis=1))
    else:
        g = csr(n, np.stack([rng.integers(0, n, 5 * n), rng.integers(0, n, 5 * n), rng.integers(0, 100, 5 * n)], axis=1))
    for delta in (1, 64, 1 << 30):
        for src in (0, n // 2, n - 1):
            check(g, min(src, g.nnodes - 1), delta)


# Vertices taken apart when they are pushed (64 edges, on graphs of more than 5
# edges a vertex) or popped (256): degrees on both sides, many in one round.
@pytest.mark.parametrize("kw", [dict(), dict(heavy_deg=40), dict(block_size=512), dict(graph_launch=True)])
def test_split_when_pushed(kw):
    rng = np.random.default_rng(5)
    n = 6000
    deg = rng.choice([0, 1, 8, 63, 64, 65, 255, 256, 257, 600], n, p=[.1, .3, .3, .05, .05, .05, .05, .04, .03, .03])
    deg[0] = 3000
    src = np.repeat(np.arange(n), deg)
    g = csr(n, np.stack([src, rng.integers(0, n, len(src)), rng.integers(0, 60, len(src))], axis=1))
    for delta in (1, 16, 1 << 20):
        check(g, 0, delta, **kw)
        check(g, 77, delta, **kw)


def test_captured_launch_takes_new_sources():
    """Replays of one captured launch, each against the oracle, with plain launches between."""
    g = CSRGraph.rmat(12, 8, seed=9)
    dev = g.copy_to_gpu()
    for src in (g.max_degree_vertex(), 1, 17, 4000):
        for graph in (True, False, True):
            print("captured", src, graph, flush=True)
            sssp_gg_main(g, dev, Options(delta=64, start_node=src, graph_launch=graph))
            dev.copy_to_cpu(g)
            assert np.array_equal(g.node_data, oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, src))
    dev.close()


def test_large_weights():
    """Distances near the end of the 31-bit range."""
    w = 2**30 - 1
    g = csr(6, [(0, 1, w), (1, 2, w), (0, 2, 2 * w), (2, 3, 1), (0, 4, 2**31 - 1), (4, 5, 7)])
    dev = g.copy_to_gpu()
    for delta in (1 << 20, 2**31 - 1):
        print("large weights", delta, flush=True)
        sssp_gg_main(g, dev, Options(delta=delta, start_node=0))
        dev.copy_to_cpu(g)
        assert np.array_equal(g.node_data, oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, 0))
    dev.close()


# A batch of graphs is packed and unpacked in tiles of 1024 edges or vertices of
# one wavefront each: members that end at and beside a tile's end, members
# without edges (first, last, in a row), many in one tile.
@pytest.mark.parametrize("members", [
    [(1, 0)], [(1, 0), (3, 1024), (1, 0)], [(1023, 1023), (1, 1), (1024, 1025), (1025, 1024)],
    [(2, 0), (5, 0), (700, 3000), (9, 0), (9, 0), (40, 255), (2500, 9000), (1, 0)], [(3, 7)] * 300 + [(1, 0)] * 3,
])
def test_union_of_members(members):
    from galoisgpu_amd.batch import sssp_graphs

    rng = np.random.default_rng(len(members))
    gs = [csr(n, np.stack([rng.integers(0, n, e), rng.integers(0, n, e), rng.integers(1, 50, e)], 1)) for n, e in members]
    srcs = [int(rng.integers(n)) for n, _ in members]
    devs = [g.copy_to_gpu() for g in gs]
    print("union", members[:8], flush=True)
    outs, _ = sssp_graphs(devs, srcs, Options(delta=20))
    for g, s, out in zip(gs, srcs, outs):
        assert np.array_equal(out, oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, s))
    for d in devs:
        d.close()
