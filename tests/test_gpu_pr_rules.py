"""PageRank at the lines of its layout's rules, against the oracle's double fixpoint:
heavy from 32, 128 or 255 in-edges by the graph's edges, vertices and mean degree;
sorting tiles of 512 vertices; the sweep with and without the table in LDS.
Tolerance 1e-4 relative, as the other PageRank tests: the truncation at epsilon 1e-6
is at most 5.7e-6, float sums of at most 4096 terms per lane add less than 1e-4."""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph
from galoisgpu_amd.apps import pagerank_into
from galoisgpu_amd.batch import DeviceArray

pytestmark = pytest.mark.gpu
RTOL = 1e-4


def check(g, block_size=None):
    print("pr rules", g.nnodes, g.nedges, flush=True)
    ref, _ = oracle.pagerank(g.row_start, g.edge_dst)
    dev = g.copy_to_gpu()
    rev, out = dev.transpose(), DeviceArray(g.nnodes * 4)
    got = []
    for _ in range(2):
        st = pagerank_into(dev, rev, out.ptr)
        got.append(out.to_numpy(np.float32, g.nnodes))
        err = np.abs(got[-1].astype(np.float64) - ref) / ref
        assert err.max() <= RTOL, (float(err.max()), int(err.argmax()))
    assert np.array_equal(got[0], got[1])  # one summation order
    if block_size:
        assert st["block_size"] == block_size
    for d in (out, rev, dev):
        d.close()


def with_in_degrees(n, degs, seed):
    rng = np.random.default_rng(seed)
    dst = np.repeat(np.arange(len(degs)), degs)
    src = rng.integers(0, n, len(dst))
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    return CSRGraph.from_arrays(row, dst[order], np.ones(len(dst)))


# At most 32768 vertices: heavy from 128; more: from 255, unless the mean is as much.
@pytest.mark.parametrize("n", [32768, 32769])
@pytest.mark.parametrize("degs", [[127] * 200 + [128] * 200 + [129] * 1300, [254] * 300 + [255] * 300 + [256] * 700,
                                  [4095, 4096, 4097] + [126, 127, 128, 255, 256] * 300])
def test_heavy_from(n, degs):
    check(with_in_degrees(n, degs, n + len(degs)))


@pytest.mark.parametrize("mean", [250, 254, 255, 260])
def test_mean_degree(mean):
    rng = np.random.default_rng(mean)
    degs = np.full(33000, mean)
    degs[:2000] = rng.integers(0, 2 * mean, 2000)
    degs[2000] += int(mean) * 33000 - degs.sum()
    check(with_in_degrees(33000, np.maximum(degs, 0), mean))


@pytest.mark.parametrize("n", [511, 512, 513, 1024, 1025, 5 * 512 + 64, 5 * 512 + 65])
def test_tiles(n):
    rng = np.random.default_rng(n)
    check(with_in_degrees(n, rng.integers(0, 31, n), n), 256)


def test_table_needs_skew():
    n = 100000
    check(with_in_degrees(n, np.full(n, 101), 3), 256)  # 40 % of the edges leave the table's vertices
    check(CSRGraph.rmat(20, 11, seed=4), 1024)
