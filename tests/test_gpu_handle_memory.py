"""Device memory of traversal handles: the arrays of dense steps (6 bytes a
vertex) belong to the handles that can take such steps."""
import ctypes
import gc

import numpy as np
import pytest
import torch

import meerkat_amd as mk
from meerkat_amd import _lib

pytestmark = pytest.mark.gpu
N = 1 << 22


def bytes_of(make):
    gc.collect()  # what earlier tests left is not freed in between
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    h = make()
    torch.cuda.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    h.Static()
    want = np.full(N, mk.INF, np.uint32)
    want[:3] = 0, 1, 2
    assert np.array_equal(h.Distances(), want)
    h.close()
    return used


@pytest.fixture(scope="module")
def graphs(gpu):
    made = []
    for mirror in (False, True):
        pool = mk.SlabPool(1 << 24)
        g = mk.DynamicGraph(N, pool, 0.7, None, weighted=True, reverse=mirror)
        g.InsertEdges(np.uint32([0, 1]), np.uint32([1, 2]), np.uint32([1, 1]))
        made.append(g)
    yield made
    for g in made:
        g.close()


def tuned(name, value, call):
    old = ctypes.c_int64()
    _lib.call("mk_tune_get", name, ctypes.byref(old))
    try:
        _lib.call("mk_tune_set", name, value)
        return call()
    finally:
        _lib.call("mk_tune_set", name, old.value)


def test_dense_arrays_only_where_used(graphs):
    plain, mirror = graphs
    full = bytes_of(lambda: mk.SSSP(plain, 0))  # takes dense steps
    none = tuned(b"persistent_steps", 0, lambda: bytes_of(lambda: mk.SSSP(plain, 0)))
    # allocations in whole MB: 6 bytes a vertex are 24 of them
    assert full - none >= 20 << 20, (full, none)
    # bottom-up BFS: two frontier bitmaps (1 MB), no dense steps
    down = bytes_of(lambda: mk.BFS(mirror, 0))
    assert down - none <= 4 << 20, (down, none)
    # near-far SSSP: three far lists, no dense steps
    far = tuned(b"sssp_far_cap", 1024, lambda: tuned(
        b"sssp_delta", 50, lambda: bytes_of(lambda: mk.SSSP(plain, 0))))
    assert far - none <= 4 << 20, (far, none)
