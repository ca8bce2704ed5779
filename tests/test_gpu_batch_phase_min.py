"""The batched kernel's smallest deferred distance of each source, against the oracle's Dijkstra.

A block reduces it in its own memory before it goes to the phase's minima, which
set the sources' thresholds in bucket mode.  The cases are each row packing (up
to 16, up to 32, more sources), each block size, a source whose column is the
last one, and phases that defer little or nearly all.
"""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph, Options
from galoisgpu_amd.batch import sssp_multi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("block_size", [256, 512, 1024])
@pytest.mark.parametrize("nsrc", [1, 2, 16, 17, 32, 33, 63, 64])
def test_phase_minima(nsrc, block_size):
    rng = np.random.default_rng(nsrc)
    n = 3000
    src = np.sort(np.concatenate([np.arange(n), rng.integers(0, n, 2 * n)]))  # no source without edges
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    g = CSRGraph.from_arrays(row, rng.integers(0, n, len(src)), rng.integers(1, 500, len(src)))
    srcs = rng.integers(0, n, nsrc)
    want = [oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, int(s)) for s in srcs]
    dev = g.copy_to_gpu()
    try:
        for delta in (20, 1500):
            for far_mode in (0, 1, 2):
                print("phase minima", nsrc, block_size, delta, far_mode, flush=True)
                d, st = sssp_multi(dev, srcs, Options(delta=delta, far_mode=far_mode, block_size=block_size))
                assert st["phases"] > 1
                for i in range(nsrc):
                    assert np.array_equal(d[:, i], want[i]), (i, delta, far_mode)
    finally:
        dev.close()
