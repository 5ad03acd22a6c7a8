"""Static triangle counts over the sorted rows against the oracle and closed
forms (exact): rows at the edges of the register, LDS and tile paths, vertices
on both sides of the bitmap's ranks, and the count over plain lists that a
bound on the scratch selects."""
import ctypes

import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import _lib, gen

pytestmark = pytest.mark.gpu


def count(n, s, d, w=None, hints=True):
    pool = mk.SlabPool(1 << 27)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s) if hints else None,
                        weighted=w is not None)
    g.InsertEdges(s, d, w)
    tc = mk.TC(g)
    tc.Static()
    first = tc.GetCount()
    tc.Static()  # again over the kept scratch
    assert tc.GetCount() == first
    return first


@pytest.mark.parametrize("k", [2, 3, 65, 66, 513, 1025, 1026, 2300])
def test_cliques(gpu, k):
    # the lowest-ranked vertex's row has k - 1 elements: 64 fill the
    # registers, 1024 the LDS tile, 512 (below the bitmap) the hash table
    a, b = np.divmod(np.arange(k * k, dtype=np.uint32), np.uint32(k))
    m = a != b
    assert count(k + 5, a[m], b[m]) == k * (k - 1) * (k - 2) // 6


@pytest.mark.parametrize("scale,weighted,hints", [(9, False, True), (15, True, True), (16, True, True),
                                                  (17, False, True), (18, False, False)])
def test_rmat(gpu, scale, weighted, hints):
    # 2^15 vertices are all within the bitmap's ranks, more are not
    n, s, d, w = gen.rmat(scale, 8, seed=scale, undirected=True, weighted=True)
    want = oracle.tc(oracle.csr(n, s, d))
    assert count(n, s, d, w if weighted else None, hints) == want


def test_no_edges_and_no_wedges(gpu):
    assert count(7, np.zeros(0, np.uint32), np.zeros(0, np.uint32), hints=False) == 0
    s = np.uint32([0, 1, 2, 3])  # two separate edges: rows of one element
    assert count(7, s, np.uint32([1, 0, 3, 2])) == 0


def test_scratch_bound_selects_plain_lists(gpu):
    n, s, d, _ = gen.rmat(15, 8, seed=4, undirected=True)
    want = oracle.tc(oracle.csr(n, s, d))
    old = ctypes.c_int64()
    _lib.call("mk_tune_get", b"tc_scratch_mb", ctypes.byref(old))
    try:
        for mb in (1, 0):
            _lib.call("mk_tune_set", b"tc_scratch_mb", mb)
            assert count(n, s, d) == want
    finally:
        _lib.call("mk_tune_set", b"tc_scratch_mb", old.value)


@pytest.mark.parametrize("weighted,hints", [(False, True), (True, True), (False, False)])
def test_batches_through_hubs(gpu, weighted, hints):
    # two hubs of several buckets (one bucket and long chains without hints)
    # joined, split and joined again within a batch: hub-hub edges, all of a
    # vertex's edges deleted, the batch's own edges closing triangles
    n, s, d, _ = gen.rmat(12, 8, seed=3, undirected=True)
    hub = np.arange(2, n - 5, dtype=np.uint32)  # the last vertices stay isolated
    a = np.r_[np.full(len(hub), 0), np.full(len(hub), 1), [0]].astype(np.uint32)
    b = np.r_[hub, hub, [1]].astype(np.uint32)
    more = np.unique(np.r_[gen.keys_of(a, b), gen.keys_of(b, a)])
    base = np.setdiff1d(gen.keys_of(s, d), more)
    S, D = gen.split_keys(base)
    allS, _ = gen.split_keys(np.union1d(base, more))
    one = np.ones(len(base) + len(more), np.uint32) if weighted else None
    pool = mk.SlabPool(1 << 27)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, allS) if hints else None,
                        weighted=weighted)
    g.InsertEdges(S, D, one[:len(S)] if weighted else None)
    tc = mk.TC(g)
    tc.Static()
    small = oracle.tc(oracle.csr(n, S, D))
    full = oracle.tc(oracle.csr(n, *gen.split_keys(np.union1d(base, more))))
    assert tc.GetCount() == small
    ms, md = (mk.device_u32(x) for x in gen.split_keys(more))
    mw = mk.device_u32(one[:len(more)]) if weighted else None
    for _ in range(2):
        g.InsertEdges(ms, md, mw)
        tc.Incremental(ms, md)
        assert tc.GetCount() == full
        g.DeleteEdges(ms, md)
        tc.Decremental(ms, md)
        assert tc.GetCount() == small
