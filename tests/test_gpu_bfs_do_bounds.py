"""A reverse graph whose sources were changed after it was wrapped: a bottom-up
level takes a source beyond the vertices as not visited.  The source used here lies
behind the visited bitmap in the same workspace buffer (two bitmaps of visited
vertices, then one of the vertices with in-edges)."""
import ctypes

import numpy as np
import pytest

from galoisgpu_amd import CSRGraph
from galoisgpu_amd._lib import check, lib
from galoisgpu_amd.apps import bfs_do_into
from galoisgpu_amd.batch import DeviceArray

pytestmark = pytest.mark.gpu


def test_source_beyond_the_vertices():
    n = 1000  # 16 words: source 1024 + k is bit k of the next bitmap
    src = np.arange(n)
    dst = np.concatenate([np.arange(1, n), [5]])  # a path, and its last vertex to vertex 5
    g = CSRGraph.from_arrays(np.arange(n + 1), dst, np.ones(n, dtype=np.int64))
    dev = g.copy_to_gpu()
    rev = dev.transpose()  # row 5 holds 4 and 999, at 4 and 5 of the array
    at = ctypes.cast(rev._g.edge_dst, ctypes.c_void_p).value + 4 * 5
    bad = np.array([1024 + 7], dtype=np.uint32)
    check(lib().lsg_dev_copy(0, ctypes.c_void_p(at), bad.ctypes.data_as(ctypes.c_void_p), 4, 0), "dev_copy")
    out = DeviceArray(4 * n)
    print("bfs_do with a source beyond the vertices", flush=True)
    bfs_do_into(dev, rev, out.ptr, 0, 2)
    assert np.array_equal(out.to_numpy(np.int32, n), src)
    for d in (out, rev, dev):
        d.close()
