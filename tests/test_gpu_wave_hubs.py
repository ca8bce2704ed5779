"""Heavy vertices (256 edges and more) on graphs of at most 5 edges a vertex,
where wavefronts go on with what they pushed: a vertex that is lowered again and
again within a round is taken apart into chunks once, so that the chunk queue
(2 E / 256 + 64 entries) holds a round's chunks.  Against the host oracle;
distances are whole numbers: equality."""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph, Options
from galoisgpu_amd.apps import bfs_gg_main, sssp_gg_main

pytestmark = pytest.mark.gpu


def csr(n, src, dst, w):
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    return CSRGraph.from_arrays(row, dst[order], w[order])


def check(g, src, delta, **kw):
    print("hubs", g.nnodes, g.nedges, src, delta, kw, flush=True)
    dev = g.copy_to_gpu()
    sssp_gg_main(g, dev, Options(delta=delta, start_node=src, **kw))
    dev.copy_to_cpu(g)
    assert np.array_equal(g.node_data, oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, src))
    bfs_gg_main(g, dev, Options(start_node=src, **kw))
    dev.copy_to_cpu(g)
    assert np.array_equal(g.node_data, oracle.bfs(g.row_start, g.edge_dst, src)[0])
    dev.close()


def chain(length, leaves, degree=1):
    """0 -> 1 -> ... -> length, each of which has an edge to the hub, every one a
    shorter way; the hub has `leaves` leaves of `degree` edges back to the chain."""
    hub = length + 1
    c = np.arange(1, length + 1)
    leaf = np.arange(hub + 1, hub + 1 + leaves)
    back = np.repeat(leaf, degree)
    src = np.concatenate([c - 1, c, np.full(leaves, hub), back])
    dst = np.concatenate([c, np.full(length, hub), leaf, 1 + back % length])
    w = np.concatenate([np.ones(length, int), 10 * (length + 2 - c), np.full(leaves, 5), np.full(len(back), 900)])
    return csr(hub + 1 + leaves, src, dst, w)


# One wavefront lowers the hub in every hop (the hub alone fills half the queue).
@pytest.mark.parametrize("length,leaves", [(8, 40000), (30, 40000), (6, 33000)])
@pytest.mark.parametrize("kw", [dict(), dict(block_size=1024), dict(graph_launch=True)])
def test_hub_lowered_along_a_chain(length, leaves, kw):
    g = chain(length, leaves)
    for delta in (1, 1000, 1 << 28):
        check(g, 0, delta, **kw)


# Degrees on both sides of a chunk, below 32769 vertices too (a block size keeps
# them off the one-workgroup kernel).
@pytest.mark.parametrize("leaves", [255, 256, 257, 512, 513, 5000])
def test_hub_sizes(leaves):
    g = chain(12, leaves, 2)
    for delta in (1, 1000):
        check(g, 0, delta, block_size=256)


def hubs_and_leaves(hubs, degree, seed, whi=255):
    """Every hub has `degree` leaves of its own, each with one edge back to a random hub."""
    rng = np.random.default_rng(seed)
    leaf = np.arange(hubs, hubs + hubs * degree)
    src = np.concatenate([np.repeat(np.arange(hubs), degree), leaf])
    dst = np.concatenate([leaf, rng.integers(0, hubs, len(leaf))])
    return csr(hubs + len(leaf), src, dst, rng.integers(1, whi + 1, len(src)))


# Many wavefronts lower the same hubs within a round.
@pytest.mark.parametrize("kw", [dict(grid_blocks=16), dict(grid_blocks=3), dict()])
@pytest.mark.parametrize("hubs,degree", [(1000, 257), (130, 600)])
def test_hubs_lowered_by_many(hubs, degree, kw):
    g = hubs_and_leaves(hubs, degree, hubs)
    for delta in (32, 1 << 20):
        check(g, 0, delta, **kw)


def test_large_hubs_and_leaves():
    check(hubs_and_leaves(6000, 257, 3), 0, 64)
