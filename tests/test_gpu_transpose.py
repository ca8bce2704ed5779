"""Reverse CSR against numpy's stable sort, exact: rows in ascending source, weights with their edges.

Sizes around the radix sort's tile (8192 edges, 1024 per wavefront), vertex
counts at each number of passes and digit width, long runs of vertices without
edges, one row or one column of every edge, and a graph without weights.
"""
import ctypes

import numpy as np
import pytest

from galoisgpu_amd import CSRGraph
from galoisgpu_amd._lib import lib

pytestmark = pytest.mark.gpu


def csr(n, src, dst, seed=1):
    order = np.argsort(src, kind="stable")  # rows keep the drawn order: unsorted, with duplicates
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    w = np.random.default_rng(seed).integers(0, 1 << 31, len(src))
    return CSRGraph.from_arrays(row, np.asarray(dst)[order], w)


def download(ptr, n, dtype):
    out = np.empty(n, dtype=dtype)
    if n:
        assert lib().lsg_dev_copy(0, out.ctypes.data_as(ctypes.c_void_p), ctypes.cast(ptr, ctypes.c_void_p),
                                  out.nbytes, 1) == 0
    return out


def check(g):
    n, m = g.nnodes, g.nedges
    src = np.repeat(np.arange(n, dtype=np.uint32), g.out_degree())
    order = np.argsort(g.edge_dst, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(g.edge_dst, minlength=n))
    dev = g.copy_to_gpu()
    rev = dev.transpose()
    try:
        assert (rev.nnodes, rev.nedges) == (n, m)
        assert np.array_equal(download(rev._g.row_start, n + 1, np.uint32), row)
        assert np.array_equal(download(rev._g.edge_dst, m, np.uint32), src[order])
        assert np.array_equal(download(rev._g.edge_data, m, np.int32), g.edge_data[order])
    finally:
        rev.close()
        dev.close()


@pytest.mark.parametrize("n", [1, 2, 3, 255, 256, 257, 65535, 65536, 65537, (1 << 20) + 1, 1 << 22])
def test_vertex_counts(n):
    rng = np.random.default_rng(n)
    print("transpose vertices", n, flush=True)
    check(csr(n, rng.integers(0, n, 30000), rng.integers(0, n, 30000)))


@pytest.mark.parametrize("m", [0, 1, 63, 1023, 1024, 1025, 8191, 8192, 8193, 100000, 1000001])
def test_edge_counts(m):
    rng = np.random.default_rng(m)
    n = 50000
    print("transpose edges", m, flush=True)
    check(csr(n, rng.integers(0, n, m), rng.integers(0, n, m)))
    check(csr(n, np.full(m, 49999), rng.integers(0, n, m)))   # one row
    check(csr(n, rng.integers(0, n, m), np.full(m, 777)))     # one column
    check(csr(n, rng.integers(0, 9, m) * 5000, rng.integers(0, n, m)))  # empty runs of 4999 rows


def test_rmat():
    check(CSRGraph.rmat(18, 16, seed=3))
