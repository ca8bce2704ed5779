"""Connected components where the single edge pass can go wrong, against the oracle's union-find, exact.

Sizes around the init tile (256 to 4096 vertices), the wavefront's 64 rows and
its 1024-edge tile; runs of vertices without edges; chains in both directions
(deep trees), a hub whose edges span many tiles, and a star of leaves whose
only edge points at the hub.
"""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph
from galoisgpu_amd.apps import cc_into
from galoisgpu_amd.batch import DeviceArray

pytestmark = pytest.mark.gpu


def csr(n, src, dst):
    src, dst = np.asarray(src, dtype=np.int64), np.asarray(dst, dtype=np.int64)
    order = np.lexsort((dst, src))
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    return CSRGraph.from_arrays(row, dst[order], np.ones(len(src)))


def check(g):
    ref, k = oracle.cc(g.row_start, g.edge_dst)
    dev, lab = g.copy_to_gpu(), DeviceArray(g.nnodes * 4)
    try:
        for _ in range(2):
            st = cc_into(dev, lab.ptr)
            assert np.array_equal(lab.to_numpy(np.int32, g.nnodes), ref)
            assert st["items"] == k
    finally:
        lab.close()
        dev.close()


@pytest.mark.parametrize("n", [2, 63, 64, 65, 255, 256, 257, 4095, 4097, 1 << 18, (1 << 21) + 3])
def test_chains(n):
    i = np.arange(n - 1)
    print("chains", n, flush=True)
    check(csr(n, i, i + 1))
    check(csr(n, i + 1, i))
    check(csr(n, np.where(i % 3 == 0, i + 1, i), np.where(i % 3 == 0, i, i + 1)))


@pytest.mark.parametrize("m", [1, 1023, 1024, 1025, 70000])
def test_empty_runs_and_hub(m):
    n = 300000  # m edges among rows that are empty for thousands of vertices
    rng = np.random.default_rng(m)
    print("runs", m, flush=True)
    check(csr(n, np.sort(rng.choice(n // 4096, m)) * 4096 + 5, rng.integers(0, n, m)))
    check(csr(n, np.full(m, n - 2), rng.choice(n, m, replace=False)))  # one row of m edges
    check(csr(n, rng.choice(n, m, replace=False), np.full(m, 77777)))  # m rows of one edge


@pytest.mark.parametrize("rows,cols", [(1, 5000), (5000, 1), (333, 777), (2048, 70)])
def test_grids(rows, cols):
    print("grid", rows, cols, flush=True)
    check(CSRGraph.grid(rows, cols, 1, 2, seed=1))
    check(CSRGraph.roadlike(rows, cols, 0.45, 0.001, 1, 2, seed=2))
