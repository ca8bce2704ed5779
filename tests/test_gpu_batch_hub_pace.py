"""The batched kernel's first threshold on graphs with a hub, against the oracle's Dijkstra.

Such graphs are a few hops deep, and what is deferred there is expanded again.
Without a schedule the second phase's threshold lies a large number of deltas on,
so that with weights to 255 a delta of 1 leaves two phases: the sources alone, and the rest.
"""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph, Options
from galoisgpu_amd.batch import sssp_multi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsrc", [1, 16, 20, 64])
@pytest.mark.parametrize("delta", [1, 32])
def test_two_phases_on_hub_graphs(nsrc, delta):
    g = CSRGraph.rmat(13, 16, seed=5)
    srcs = np.random.default_rng(nsrc).integers(0, g.nnodes, nsrc)
    dev = g.copy_to_gpu()
    try:
        print("hub pace", nsrc, delta, flush=True)
        d, st = sssp_multi(dev, srcs, Options(delta=delta))
    finally:
        dev.close()
    for i, s in enumerate(srcs):
        assert np.array_equal(d[:, i], oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, int(s))), i
    assert st["phases"] <= 2
