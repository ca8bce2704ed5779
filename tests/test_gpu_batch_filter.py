"""The batched kernel's edge filter against the oracle's Dijkstra, exact in every column.

The filter tests an edge against a bound per vertex and is used on graphs with
a hub, once three quarters of the sources have reached it.  The cases are
where that can go wrong: few and many sources, sources that never reach the
hub, weights of zero and near INT_MAX (sums that saturate), every far mode,
chunk sizes at both ends, graphs whose size is no multiple of a wavefront.
"""
import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph, Options
from galoisgpu_amd.batch import sssp_multi

pytestmark = pytest.mark.gpu

INT_MAX = 0x7FFFFFFF


def hub_graph(n, seed, whi, wlo=0):
    """A hub with edges to and from a third of the vertices, random edges besides, and a part cut off from the hub."""
    rng = np.random.default_rng(seed)
    core = n - n // 8
    spokes = rng.choice(core, core // 3, replace=False)
    src = np.concatenate([np.full(len(spokes), 7), spokes, rng.integers(0, core, 4 * n), rng.integers(core, n, n // 4)])
    dst = np.concatenate([spokes, np.full(len(spokes), 7), rng.integers(0, core, 4 * n), rng.integers(core, n, n // 4)])
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    w = rng.integers(wlo, whi, len(src), endpoint=True)
    return CSRGraph.from_arrays(row, dst[order], w)


def check(g, srcs, **kw):
    dev = g.copy_to_gpu()
    try:
        d, st = sssp_multi(dev, srcs, Options(**kw))
    finally:
        dev.close()
    for i, s in enumerate(srcs):
        assert np.array_equal(d[:, i], oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, int(s))), (i, s, kw)
    return st


@pytest.mark.parametrize("n,nsrc,whi", [(1000, 1, 255), (4097, 5, 255), (20011, 33, 1), (20011, 64, 255),
                                        (3001, 64, INT_MAX), (65537, 17, 1 << 28)])
def test_hub_graphs(n, nsrc, whi):
    g = hub_graph(n, n + nsrc, whi)
    srcs = np.random.default_rng(nsrc).integers(0, n, nsrc)  # about an eighth cannot reach the hub
    print("filter", n, nsrc, whi, flush=True)
    check(g, srcs, delta=1 << 30)


@pytest.mark.parametrize("far_mode", [0, 1, 2])
@pytest.mark.parametrize("heavy_deg", [8, 64, 700])
def test_modes_and_chunks(far_mode, heavy_deg):
    g = CSRGraph.rmat(13, 12, seed=3)
    srcs = np.random.default_rng(far_mode).integers(0, g.nnodes, 40)
    print("filter modes", far_mode, heavy_deg, flush=True)
    check(g, srcs, delta=64, far_mode=far_mode, heavy_deg=heavy_deg, block_size=256)


def test_most_sources_cut_off_from_the_hub():
    g = hub_graph(8000, 5, 100)
    cut = np.arange(7000 + 8, 7000 + 40)
    check(g, np.concatenate([cut, [1, 2, 3]]), delta=1 << 30)


def test_more_work_units_than_wavefronts():
    # rounds of more than 4096 x 16 items: tickets, group helping, staged heavy items
    g = CSRGraph.rmat(18, 8, seed=9)
    srcs = np.random.default_rng(1).integers(0, g.nnodes, 12)
    st = check(g, srcs, delta=1 << 30, block_size=256, heavy_deg=16)
    assert st["items"] > 4096 * 16


@pytest.mark.parametrize("n", [1500, 3000, 3001, 3016, 5004, 20011])
def test_bounds_of_an_earlier_call_are_not_seen(n):
    """Vertices 0 to 15 lie beside the other arrays' last vertices in the bounds of the second and third
    sweep.  Seen from `a` they are near and the hub is far, seen from the other sources the reverse:
    a bound left over from the call before would cut them off."""
    rng = np.random.default_rng(n)
    hub, chain, first = 20, 60, 16
    a = first + 4 + chain
    core = np.arange(a + 1, n)
    spokes = rng.choice(core, len(core) // 3, replace=False)
    links = np.arange(first + 4, a)                        # hub+1 ... a: a chain that only ends at a
    src = np.concatenate([np.full(len(spokes), hub), spokes, rng.choice(core, 8 * n),
                          rng.choice(core, 9000), [core[5]], links[1:], [a - 1], np.full(16, a), [a]])
    dst = np.concatenate([spokes, np.full(len(spokes), hub), rng.choice(core, 8 * n),
                          rng.integers(n - 16, n, 9000), [links[1]], links[1:] + 1, [a], np.arange(16), [hub]])
    w = rng.integers(1, 255, len(src))
    w[-1] = 1000000
    order = np.argsort(src, kind="stable")
    row = np.zeros(n + 1, dtype=np.int64)
    row[1:] = np.cumsum(np.bincount(src, minlength=n))
    g = CSRGraph.from_arrays(row, dst[order], w[order])
    dev = g.copy_to_gpu()
    others = [int(x) for x in rng.choice(core, 4)]
    ref = {s: oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, s) for s in [a] + others}
    for s in others * 3:
        for srcs in ([a], [s]):
            print("bounds of an earlier call", n, srcs, flush=True)
            d, _ = sssp_multi(dev, srcs, Options(delta=1 << 30))
            assert np.array_equal(d[:, 0], ref[srcs[0]]), srcs
    dev.close()


@pytest.mark.parametrize("blocks", [1, 3, 15, 16, 17, 31, 33, 250])
def test_every_unit_is_taken(blocks):
    """Grids that the ticket groups do not divide evenly, with fewer and more units than wavefronts."""
    g = CSRGraph.rmat(12, 8, seed=4)
    srcs = np.random.default_rng(blocks).integers(0, g.nnodes, 20)
    for block_size in (256, 1024):
        print("units", blocks, block_size, flush=True)
        check(g, srcs, delta=40, grid_blocks=blocks, block_size=block_size)
        check(CSRGraph.grid(40, 60, seed=blocks), [3, 700], delta=64, grid_blocks=blocks, block_size=block_size)


@pytest.mark.parametrize("whi", [1, 100, 60000, 1 << 24])
@pytest.mark.parametrize("delta", [1, 32, 1 << 28])
def test_paced_threshold(whi, delta):
    """Steps of delta that grow from phase to phase, on graphs with and without a hub."""
    print("paced", whi, delta, flush=True)
    check(hub_graph(3001, whi, whi), [0, 1, 7, 2000, 2999], delta=delta)
    check(CSRGraph.grid(60, 41, 1, whi, seed=3), [0, 17, 2459], delta=delta)


@pytest.mark.parametrize("nsrc", [1, 2, 15, 16, 17, 31, 32, 33])
def test_packed_rows(nsrc):
    """Source counts on both sides of each row packing, every far mode, chunks and light items."""
    g = CSRGraph.rmat(12, 10, seed=nsrc)
    live = np.flatnonzero(np.diff(g.row_start.astype(np.int64)))  # each source keeps its column
    srcs = np.random.default_rng(nsrc).choice(live, nsrc, replace=False)
    for far_mode in (0, 1, 2):
        for heavy_deg in (8, 64, 4000):
            print("packed", nsrc, far_mode, heavy_deg, flush=True)
            check(g, srcs, delta=40, far_mode=far_mode, heavy_deg=heavy_deg)
    check(hub_graph(4001, nsrc, INT_MAX), srcs, delta=1 << 30)
    check(CSRGraph.grid(50, 60, 1, 100, seed=nsrc), np.arange(nsrc) * 90, delta=64)
