"""Captured single-source launches after other calls have moved the buffer that holds the seeds.

A captured launch reads its seeds from a workspace buffer that building a reverse CSR
and batched runs use too, and grow.  A replay made for the same graph and output must
not read where the buffer was before: each call is compared with the oracle.
"""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph, Options
from galoisgpu_amd.apps import bfs_into, sssp_into
from galoisgpu_amd.batch import DeviceArray, sssp_graphs, sssp_multi

pytestmark = pytest.mark.gpu


def transpose_of(n):
    g = CSRGraph.grid(n, n, seed=n)
    dev = g.copy_to_gpu()
    dev.transpose().close()
    dev.close()


def batch():
    dev = CSRGraph.grid(20, 20, seed=1).copy_to_gpu()
    sssp_multi(dev, [0, 1, 2], Options(delta=32))
    dev.close()


def graphs():
    devs = [CSRGraph.grid(5, 5, seed=i).copy_to_gpu() for i in range(40)]
    sssp_graphs(devs, [0] * len(devs), Options(delta=32))
    for d in devs:
        d.close()


@pytest.mark.parametrize("between", [[batch], [graphs], [lambda: transpose_of(16)],
                                     [lambda n=n: transpose_of(n) for n in (40, 200, 700)]],
                         ids=["batch", "graphs", "transpose", "transposes"])
def test_replays_after_the_seeds_have_moved(between):
    from galoisgpu_amd._lib import check, lib

    check(lib().lsg_workspace_release(0), "workspace_release")  # the buffer begins at its smallest
    g = CSRGraph.rmat(12, 8, seed=4)
    n = g.nnodes
    dev = g.copy_to_gpu()
    out = DeviceArray(n * 4)
    srcs = [int(s) for s in np.random.default_rng(len(between)).integers(0, n, 1 + len(between))]
    try:
        for i, s in enumerate(srcs):
            for kw in (dict(), dict(far_mode=1)):
                print("capture seeds", i, s, kw, flush=True)
                sssp_into(dev, out.ptr, Options(delta=32, start_node=s, graph_launch=True, **kw))
                assert np.array_equal(out.to_numpy(np.int32, n), oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, s))
                bfs_into(dev, out.ptr, Options(start_node=s, graph_launch=True, **kw))
                assert np.array_equal(out.to_numpy(np.int32, n), oracle.bfs(g.row_start, g.edge_dst, s)[0])
            if i < len(between):
                between[i]()
    finally:
        out.close()
        dev.close()
