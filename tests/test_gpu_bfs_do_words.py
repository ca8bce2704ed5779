"""Bottom-up BFS levels deal the bitmap's words of 64 vertices to wavefronts, a
unit's words as far apart as there are units: sizes at the edges of a word, of a
unit of 16 words and of the launch (one word each for 1024 wavefronts, two blocks
a CU from 2^18 vertices), with neighbouring hubs.  Levels against the host oracle."""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph
from galoisgpu_amd.apps import bfs_do_into
from galoisgpu_amd.batch import DeviceArray

pytestmark = pytest.mark.gpu


def graph(n, hubs):
    """Vertices below `hubs` are joined to many others, both ways; the others to two of them; some random edges."""
    rng = np.random.default_rng(n)
    hubs = max(1, min(hubs, n // 2))
    v = np.arange(hubs, n)
    p, q = rng.integers(0, hubs, len(v)), rng.integers(0, hubs, len(v))
    x = rng.integers(0, n, (2, n))
    src = np.concatenate([v, p, q, x[0]])
    dst = np.concatenate([p, v, v, x[1]])
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    return CSRGraph.from_arrays(row, dst[order], np.ones(len(src), dtype=np.int64))


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1024, 1025, 16 * 64, 65535, 65536, 65537, (1 << 18) - 1, 1 << 18,
                               (1 << 18) + 1, 1024 * 1024 + 64, 16 * 64 * 1024 + 1])
def test_sizes(n):
    g = graph(n, 300)
    ref, _ = oracle.bfs(g.row_start, g.edge_dst, n - 1)
    dev = g.copy_to_gpu()
    rev = dev.transpose()
    out = DeviceArray(4 * n)
    for direction in (2, 0, 1):
        print("bfs_do words", n, direction, flush=True)
        bfs_do_into(dev, rev, out.ptr, n - 1, direction)
        assert np.array_equal(out.to_numpy(np.int32, n), ref)
    for d in (out, rev, dev):
        d.close()
