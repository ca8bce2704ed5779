"""What a call whose grid barrier gives up says of where it was.

The limit is set from the host; every wavefront still leaves the kernel.  A vertex
of 400,000 edges, not taken apart, keeps one wavefront busy for milliseconds in a round
that the others wait for, a chain of vertices after the source: with a limit between the
two the round that the text names is one after the first.
"""
import re

import numpy as np
import pytest

import oracle
from galoisgpu_amd import CSRGraph, LsgError
from galoisgpu_amd.apps import sssp

pytestmark = pytest.mark.gpu


def test_timeout_names_the_round(monkeypatch):
    chain, leaves = 4, 400_000
    n = chain + 1 + leaves
    row = np.concatenate([np.arange(chain + 1), np.full(n - chain, chain + leaves)])
    row[chain] = chain
    dst = np.concatenate([np.arange(1, chain + 1), np.arange(chain + 1, n)])
    w = np.full(len(dst), 100)
    g = CSRGraph.from_arrays(row, dst, w)
    monkeypatch.setenv("LSG_BARRIER_TIMEOUT_S", "0.0005")
    print("timeout text", flush=True)
    with pytest.raises(LsgError) as e:
        sssp(g, 0, 32, heavy_deg=1 << 24)
    assert e.value.name == "LSG_ERR_TIMEOUT"
    m = re.search(r"round (\d+) phase (\d+)", str(e.value))
    assert m and int(m.group(1)) > 1 and int(m.group(2)) >= 1, str(e.value)
    monkeypatch.delenv("LSG_BARRIER_TIMEOUT_S")
    d, _ = sssp(g, 0, 32, heavy_deg=1 << 24)
    assert np.array_equal(d, oracle.dijkstra(g.row_start, g.edge_dst, g.edge_data, 0))
