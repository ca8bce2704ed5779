"""Low-degree graphs whose frontier grows by factors (random, skewed, trees, hubs
with leaves), where the wavefront kernel's rounds turn wide: against the host
oracle at sizes on both sides of the one-workgroup kernel's, of a round of one
block (512 items) and of the rounds that still go on (8192 and 16384 items)."""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph, Options
from galoisgpu_amd.apps import bfs_gg_main, sssp_gg_main

pytestmark = pytest.mark.gpu
INF = 2**31 - 1


def csr(n, src, dst, whi, rng):
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    return CSRGraph.from_arrays(row, dst[order], rng.integers(1, whi + 1, len(src)))


def graph(kind, n, whi=255):
    rng = np.random.default_rng(n)
    if kind == "rmat":  # at most 5 edges a vertex
        g = CSRGraph.rmat(int(n).bit_length() - 1, 5, 0.57, 0.19, 0.19, 1, whi, seed=2)
        assert g.nedges <= 5 * g.nnodes
        return g
    if kind == "uniform":
        src, dst = np.repeat(np.arange(n), 4), rng.integers(0, n, 4 * n)
    elif kind in ("random tree", "tree"):
        v = np.arange(1, n)
        p = (rng.random(n - 1) * v).astype(np.int64) if kind == "random tree" else (v - 1) // 16
        src, dst = np.concatenate([v, p]), np.concatenate([p, v])
    elif kind == "bipartite":  # 200 hubs, every other vertex joined to two of them
        v = np.arange(200, n)
        p, q = rng.integers(0, 200, n - 200), rng.integers(0, 200, n - 200)
        src, dst = np.concatenate([v, p, q, v]), np.concatenate([p, v, v, q])
    else:  # a road network behind a hub: growth that says nothing
        g = CSRGraph.roadlike(n // 256, 256, 0.1, 0.001, 1, 1000, seed=1)
        m, e = g.nnodes, g.nedges
        to = rng.choice(m, 3000, replace=False)
        src = np.concatenate([np.repeat(np.arange(m), np.diff(g.row_start.astype(np.int64))), np.full(3000, m)])
        return csr(m + 1, src, np.concatenate([g.edge_dst, to]), 1000, rng)
    return csr(n, src, dst, whi, rng)


@pytest.mark.parametrize("kind", ["rmat", "uniform", "random tree", "tree", "bipartite", "hub and road"])
@pytest.mark.parametrize("n", [4096, 40000, 300000])
def test_against_the_oracle(kind, n):
    g = graph(kind, n)
    src = g.max_degree_vertex()
    dev = g.copy_to_gpu()
    for kw in (dict(block_size=256), dict(grid_blocks=5, block_size=256), dict(graph_launch=True)):
        for delta in (1, 32, 10000):
            print("wide", kind, n, delta, kw, flush=True)
            sssp_gg_main(g, dev, Options(delta=delta, start_node=src, **kw))
            dev.copy_to_cpu(g)
            assert np.array_equal(g.node_data, oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, src))
        bfs_gg_main(g, dev, Options(start_node=src, **kw))
        dev.copy_to_cpu(g)
        assert np.array_equal(g.node_data, oracle.bfs(g.row_start, g.edge_dst, src)[0])
    dev.close()


def test_wide_levels_are_expanded_once():
    """BFS of a random graph: only rounds of up to 8192 of its 400,000 vertices go
    on beyond their level, so that at most a quarter is expanded twice."""
    g = graph("uniform", 400000)
    dev = g.copy_to_gpu()
    ref, _ = oracle.bfs(g.row_start, g.edge_dst, 0)
    reached = np.count_nonzero(ref != INF)
    for _ in range(3):
        st = bfs_gg_main(g, dev, Options(start_node=0))
        print("items", st["items"], "reached", reached, flush=True)
        assert reached <= st["items"] <= 1.25 * reached
    dev.close()
