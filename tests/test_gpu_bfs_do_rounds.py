"""The levels of the direction-optimising BFS at the edges of its rounds, against
the oracle's BFS, under every direction policy.  Levels are whole numbers: equality."""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph
from galoisgpu_amd.apps import BFS_AUTO, BFS_BOTTOM_UP, BFS_TOP_DOWN, bfs_do_into
from galoisgpu_amd.batch import DeviceArray

pytestmark = pytest.mark.gpu


def csr(n, src, dst):
    src, dst = np.asarray(src, dtype=np.int64), np.asarray(dst, dtype=np.int64)
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    return CSRGraph.from_arrays(row, dst[order])


def check(g, srcs):
    dev = g.copy_to_gpu()
    rev = dev.transpose()
    lv = DeviceArray(g.nnodes * 4)
    for s in srcs:
        ref, _ = oracle.bfs(g.row_start, g.edge_dst, int(s))
        top = int(ref[ref != 2**31 - 1].max())
        for d in (BFS_AUTO, BFS_TOP_DOWN, BFS_BOTTOM_UP):
            print("bfs_do rounds", g.nnodes, g.nedges, s, d, flush=True)
            st = bfs_do_into(dev, rev, lv.ptr, int(s), d)
            assert np.array_equal(lv.to_numpy(np.int32, g.nnodes), ref), (s, d)
            assert st["iterations"] == top
            assert d != BFS_TOP_DOWN or st["near_iters"] == 0
    lv.close()
    rev.close()
    dev.close()
    return st


# Levels of one block (up to 512 vertices), its piles (1024), staged vertices
# (256 a wavefront), heavy vertices (256 edges) found in either kind of level.
@pytest.mark.parametrize("degrees", [(1,), (255,), (256, 1), (257, 1, 1), (8, 64, 1), (16, 64), (4, 300, 1), (33, 34, 2),
                                     (300, 3, 3), (2, 1500, 1), (70, 257, 1), (3, 300, 4)])
def test_trees(degrees):
    src, dst, level, n = [], [], [0], 1
    for d in degrees:
        nxt = list(range(n, n + d * len(level)))
        src += [u for u in level for _ in range(d)]
        dst += nxt
        n += len(nxt)
        level = nxt
    # a path behind the last level, and edges back
    src += [level[-1]] + list(range(n, n + 5)) + list(range(1, n))
    dst += list(range(n, n + 6)) + [0] * (n - 1)
    check(csr(n + 6, src, dst), [0, n])


# Bitmap words and units: sizes beside multiples of 64; unreachable parts.
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 1023, 1025, 65537, 200001])
def test_sizes(n):
    rng = np.random.default_rng(n)
    m = 12 * n
    src = np.concatenate([rng.integers(0, max(1, n - n // 4), m), np.full(min(n, 5000), 0)])
    dst = np.concatenate([rng.integers(0, n, m), rng.integers(0, n, min(n, 5000))])
    check(csr(n, src, dst), [0, n - 1, n // 2])


@pytest.mark.parametrize("rows", [64, 65, 300, 5000])
def test_long_in_rows(rows):
    """Vertices whose many in-edges come from unreached vertices, except a last one or none."""
    rng = np.random.default_rng(rows)
    n, far = 20000, 9000                       # vertices from `far` on are not reached
    src = [np.full(6000, 0), rng.integers(1, 6000, 60000), np.arange(6000, 6040), rng.integers(far, n, 40000)]
    dst = [np.arange(1, 6001), rng.integers(1, 6000, 60000), np.arange(6001, 6041), rng.integers(far, n, 40000)]
    for i in range(40):                        # long rows, half of them found by their last in-edge
        src += [rng.integers(far, n, rows), [5999 if i % 2 else n - 1]]
        dst += [np.full(rows, 7000 + i), [7000 + i]]
    src, dst = np.concatenate(src), np.concatenate(dst)
    g = csr(n, src, dst)
    check(g, [0])
