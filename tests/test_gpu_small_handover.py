"""Where the one-workgroup kernel hands a wide frontier to the whole grid: rounds
of 4096 vertices and more, vertices of 256 edges above 8192 vertices, a source of
more edges than a list holds.  Against the host oracle; the grid that the call
reports tells which kernel ended it."""
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


def fans(fan, width, n, seed=1):
    """0 has ceil(width / fan) children of `fan` children each, `width` in all, and a tail of single vertices to n."""
    rng = np.random.default_rng(seed)
    k = -(-width // fan)
    leaf = 1 + k + np.arange(width)
    tail = np.arange(1 + k + width - 1, n - 1)
    src = np.concatenate([np.zeros(k, int), 1 + np.arange(width) // fan, tail])
    dst = np.concatenate([1 + np.arange(k), leaf, tail + 1])
    extra = rng.integers(0, n, (2, n))  # cross edges, which lower distances again
    src, dst = np.concatenate([src, extra[0]]), np.concatenate([dst, extra[1]])
    return csr(n, src, dst, rng.integers(0, 60, len(src)))


def check(g, src, handed=None):
    dev = g.copy_to_gpu()
    for delta in (1, 64, 1 << 28):
        print("handover", g.nnodes, g.nedges, src, delta, flush=True)
        st = sssp_gg_main(g, dev, Options(delta=delta, start_node=src))
        dev.copy_to_cpu(g)
        assert np.array_equal(g.node_data, oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, src))
        if handed:
            assert st["grid_blocks"] > 1
    st = bfs_gg_main(g, dev, Options(start_node=src))
    dev.copy_to_cpu(g)
    ref, _ = oracle.bfs(g.row_start, g.edge_dst, src)
    assert np.array_equal(g.node_data, ref)
    assert st["iterations"] == ref[ref != 2**31 - 1].max() + 1
    if handed is not None:
        assert (st["grid_blocks"] > 1) == handed
    dev.close()


@pytest.mark.parametrize("width", [1000, 4000, 4096, 4097, 9000, 32000])
def test_round_width(width):
    n = max(9000, width + 700)
    check(fans(64, width, n), 0, True if width > 5000 else False if width < 2000 else None)


@pytest.mark.parametrize("fan,n", [(240, 9000), (253, 9000), (256, 9000), (300, 32768), (256, 8192), (256, 8193)])
def test_hub(fan, n):
    g = fans(fan, 3 * fan, n)  # (cross edges add to the fans)
    check(g, 0, n > 8192 and int(np.diff(g.row_start.astype(np.int64)).max()) >= 256)


@pytest.mark.parametrize("n,handed", [(200, False), (4097, False), (4098, True), (8192, True), (8193, True), (32768, True)])
def test_star(n, handed):
    v = np.arange(1, n)
    z = np.zeros(n - 1, int)
    check(csr(n, np.concatenate([v, z]), np.concatenate([z, v]), 1 + np.arange(2 * (n - 1)) % 50), 0, handed)


@pytest.mark.parametrize("n", [20000, 32768])
def test_from_a_leaf(n):
    """The wide rounds come late, behind a path."""
    g = fans(40, n // 2, n)
    check(g, n - 1)
    check(g, n // 2)
