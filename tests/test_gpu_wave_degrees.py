"""Graphs with vertices of more edges than a round of one block takes.

From 16 edges on such a vertex sends its round to the whole grid, on low-degree graphs
one item a unit.  The cases have degrees on both sides of that, in the first rounds and in
the middle of a traversal, rounds of every size between the block's and the grid's, and,
on low-degree graphs, more than 32,768 vertices (fewer run in one workgroup).  Against
the oracle, exact.
"""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph
from galoisgpu_amd.apps import bfs, sssp

pytestmark = pytest.mark.gpu

N = 40_000


def both(n, u, v, seed, whi=255):
    src, dst = np.concatenate([u, v]), np.concatenate([v, u])
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    w = np.random.default_rng(seed).integers(1, whi, len(src), endpoint=True)
    return CSRGraph.from_arrays(row, dst[order], w)


def tree(k):
    v = np.arange(1, N)
    return both(N, v, (v - 1) // k, k)


def hubs(k):
    rng = np.random.default_rng(k)
    v = np.arange(k, N)
    return both(N, np.concatenate([v, v]), rng.integers(0, k, 2 * len(v)), k)


def comb(deg):
    """A path with a bush of `deg` leaves at every 50th vertex, rounds of one block in between."""
    spine = np.arange(N // 2)
    at = spine[::50]
    u = np.repeat(at, deg)
    leaf = N // 2 + np.arange(len(u)) % (N - N // 2)
    return both(N, np.concatenate([spine[:-1], u]), np.concatenate([spine[1:], leaf]), deg, 60)


def check(g, src):
    want, levels = oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, src), oracle.bfs(g.row_start, g.edge_dst, src)[0]
    for delta in (1, 32, 10000):
        d, _ = sssp(g, src, delta)
        assert np.array_equal(d, want), delta
    d, _ = bfs(g, src)
    assert np.array_equal(d, levels)


@pytest.mark.parametrize("k", [13, 14, 15, 16, 31, 64, 200, 254, 255])
def test_trees(k):
    print("tree", k, flush=True)
    check(tree(k), 1)


@pytest.mark.parametrize("k", [300, 1000, 5000])
def test_leaves_of_two_hubs(k):
    print("hubs", k, flush=True)
    check(hubs(k), 7)


@pytest.mark.parametrize("deg", [10, 12, 13, 14, 40, 300])
def test_bushes_on_a_path(deg):
    print("comb", deg, flush=True)
    check(comb(deg), 3)


@pytest.mark.parametrize("n", [300, 3000])
@pytest.mark.parametrize("deg", [8, 15, 16, 17, 40])
def test_every_vertex_of_one_degree(n, deg):
    rng = np.random.default_rng(deg)
    g = CSRGraph.from_arrays(np.arange(n + 1) * deg, rng.integers(0, n, n * deg), rng.integers(0, 100, n * deg))
    print("uniform", n, deg, flush=True)
    check(g, 5)
