"""lsg_opts.heavy_deg on single-source calls: how many chunks a vertex is taken apart into.

A value below the block size is raised to it.  One vertex of 5000 edges to vertices
without any is expanded once, so that the count is exact; the distances of a graph with
degrees on both sides of the values are the oracle's.
"""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph
from galoisgpu_amd.apps import bfs, sssp

pytestmark = pytest.mark.gpu

CASES = [(256, 1), (256, 40), (256, 256), (256, 257), (256, 1024), (512, 300), (512, 513), (1024, 1000), (1024, 5000),
         (256, 5001)]


@pytest.mark.parametrize("block,heavy", CASES)
def test_chunks_of_one_vertex(block, heavy):
    n = 5001
    g = CSRGraph.from_arrays(np.concatenate([[0], np.full(n, 5000)]), np.arange(1, n), np.arange(1, n))
    for run in (lambda: sssp(g, 0, 1 << 20, block_size=block, heavy_deg=heavy),
                lambda: bfs(g, 0, block_size=block, heavy_deg=heavy)):
        print("heavy_deg", block, heavy, flush=True)
        _, st = run()
        eff = max(block, heavy)
        assert st["heavy_chunks"] == (-(-5000 // eff) if 5000 >= eff else 0)


@pytest.mark.parametrize("block,heavy", CASES)
def test_degrees_on_both_sides(block, heavy):
    rng = np.random.default_rng(heavy)
    n, eff = 4000, max(block, heavy)
    deg = rng.choice([1, 8, 63, 64, eff - 1, eff, eff + 1, 2 * eff], n,
                     p=[.4, .4, .07, .07, .015, .015, .015, .015])
    deg[0] = 3 * eff
    src = np.repeat(np.arange(n), deg)
    g = CSRGraph.from_arrays(np.concatenate([[0], np.cumsum(deg)]), rng.integers(0, n, len(src)),
                             rng.integers(0, 60, len(src)))
    want = oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, 0)
    for delta in (1, 16, 1 << 20):
        print("heavy_deg", block, heavy, delta, flush=True)
        d, _ = sssp(g, 0, delta, block_size=block, heavy_deg=heavy)
        assert np.array_equal(d, want), delta
