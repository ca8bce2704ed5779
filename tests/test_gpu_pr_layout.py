"""PageRank on graphs whose in-degrees sit at the edges of its layout, against the oracle's double fixpoint.

Tolerance: an iteration contracts the error by alpha = 0.85 and the last one
moved no rank by more than 1e-6 of itself, so the truncation is at most 1e-6 *
0.85 / 0.15 = 5.7e-6; float sums of at most 4096 terms per lane or chunk add at
most 4096 * 2^-24 = 2.5e-4 in the worst case, of random sign in practice, over
the same geometric series.  RTOL 1e-4 is what the other PageRank tests use.
"""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph
from galoisgpu_amd.apps import pagerank_into
from galoisgpu_amd.batch import DeviceArray

pytestmark = pytest.mark.gpu
RTOL = 1e-4


def check(g, runs=2):
    ref, _ = oracle.pagerank(g.row_start, g.edge_dst)
    dev = g.copy_to_gpu()
    rev, out = dev.transpose(), DeviceArray(g.nnodes * 4)
    try:
        got = []
        for _ in range(runs):
            pagerank_into(dev, rev, out.ptr)
            got.append(out.to_numpy(np.float32, g.nnodes))
            err = np.abs(got[-1].astype(np.float64) - ref) / ref
            assert err.max() <= RTOL, (float(err.max()), int(err.argmax()))
        assert all(np.array_equal(x, got[0]) for x in got)  # one summation order
    finally:
        out.close()
        rev.close()
        dev.close()


def with_in_degrees(n, degs, seed):
    """Vertex i < len(degs) has in-degree degs[i], from random sources."""
    rng = np.random.default_rng(seed)
    dst = np.repeat(np.arange(len(degs)), degs)
    src = rng.integers(0, n, len(dst))
    order = np.lexsort((dst, src))
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    return CSRGraph.from_arrays(row, dst[order], np.ones(len(dst)))


@pytest.mark.parametrize("degs", [
    [1], [31], [32], [254], [255], [256], [4096], [4097], [8193],
    [31] * 65, [32] * 65, [254] * 64 + [255] * 3, [31, 32] * 40 + [0, 1] * 40,
    list(range(0, 300)), [5000] + [7] * 1000, [255] * 70 + [33] * 70 + [1] * 5000,
])
def test_in_degrees(degs):
    print("pr in-degrees", degs[:4], len(degs), flush=True)
    check(with_in_degrees(max(9000, 2 * len(degs)), degs, len(degs)))


@pytest.mark.parametrize("n", [1, 64, 4095, 4096, 4097, 12289])
def test_sizes_without_hubs(n):
    rng = np.random.default_rng(n)
    print("pr sizes", n, flush=True)
    check(with_in_degrees(n, rng.integers(0, 9, n), n))


def test_ranks_in_lds():
    # enough edges, hubs and vertices for the sweep that keeps the hubs' contributions in LDS
    g = CSRGraph.rmat(20, 11, seed=4)
    assert g.nedges >= 10000000
    check(g, runs=2)
