"""Device memory of triangle counting: batches whose edges' buckets are more
than the bound on work items (worked in windows, the count exact), and
the bound on the static count's scratch, which the fallback gives back."""
import ctypes
import gc

import numpy as np
import pytest
import torch

import meerkat_amd as mk
from meerkat_amd import _lib, gen

pytestmark = pytest.mark.gpu


def held(call):
    """Bytes of device memory that `call` leaves allocated."""
    gc.collect()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    call()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("weighted,hubs,share", [(False, 300, 0.325), (True, 200, 0.4)])
def test_batch_of_hub_edges(gpu, weighted, hubs, share):
    # hubs of some 13,000 / 16,000 leaves (295 / 740 buckets); the batch joins
    # all of them: 13 / 15 million (edge, bucket) pairs, against 4.2 million
    # items of 8 bytes
    leaves = 40_000
    n = hubs + leaves
    a = np.random.default_rng(hubs).random((hubs, leaves)) < share
    h, leaf = (x.astype(np.uint32) for x in np.nonzero(a))
    leaf += np.uint32(hubs)
    i, j = (x.astype(np.uint32) for x in np.nonzero(~np.eye(hubs, dtype=bool)))
    s, d = np.r_[h, leaf], np.r_[leaf, h]
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, np.r_[s, i]), weighted=weighted)
    g.InsertEdges(s, d, np.ones(len(s), np.uint32) if weighted else None)
    tc = mk.TC(g)
    tc.Static()
    assert tc.GetCount() == 0
    common = a.astype(np.float32) @ a.T.astype(np.float32)  # whole numbers below 2^24
    want = hubs * (hubs - 1) * (hubs - 2) // 6 + int(np.triu(common, 1).astype(np.int64).sum())
    bi, bj = mk.device_u32(i), mk.device_u32(j)
    bw = mk.device_u32(np.ones(len(i), np.uint32)) if weighted else None
    for _ in range(2):
        g.InsertEdges(bi, bj, bw)
        used = held(lambda: tc.Incremental(bi, bj))
        assert tc.GetCount() == want
        assert used <= 48 << 20, used  # items 32 MB, the edges' arrays 4 MB
        g.DeleteEdges(bi, bj)
        tc.Decremental(bi, bj)
        assert tc.GetCount() == 0


@pytest.mark.parametrize("edges,mb", [(1000, 8), (4_000_000, 64)])
def test_static_scratch_within_its_bound(gpu, edges, mb):
    # 2^20 vertices: the sorted lists' per-vertex arrays (48 bytes) alone
    # exceed 8 MB; with 8M directed entries they and the rows exceed 64 MB.
    # The plain lists take 16 bytes a vertex and 4 an undirected edge.
    n = 1 << 20
    s, d, _ = gen.insert_batch(None, n // 2, edges, seed=edges)
    keys = np.unique(np.r_[gen.keys_of(s, d), gen.keys_of(d, s)])
    S, D = gen.split_keys(keys)
    # and a clique of 60 on ids that the edges above do not touch
    a, b = np.divmod(np.arange(3600, dtype=np.uint32), np.uint32(60))
    m = a != b
    A, B = a[m] + np.uint32(n - 60), b[m] + np.uint32(n - 60)
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, np.r_[S, A]))
    g.InsertEdges(np.r_[S, A], np.r_[D, B])
    old = ctypes.c_int64()
    _lib.call("mk_tune_get", b"tc_scratch_mb", ctypes.byref(old))
    free, tc = mk.TC(g), mk.TC(g)
    try:
        _lib.call("mk_tune_set", b"tc_scratch_mb", 0)
        free.Static()
        want = free.GetCount()
        assert want >= 60 * 59 * 58 // 6
        _lib.call("mk_tune_set", b"tc_scratch_mb", mb)
        for handle in (tc, free):  # a fresh one, and one that holds more
            used = held(handle.Static)
            assert handle.GetCount() == want
            # plain lists 16 MB + 4 B an edge; four allocations rounded to 2 MB
            assert used <= (24 << 20) + 4 * edges, used
        _lib.call("mk_tune_set", b"tc_scratch_mb", 256)
        assert held(tc.Static) <= 256 << 20
        assert tc.GetCount() == want
    finally:
        _lib.call("mk_tune_set", b"tc_scratch_mb", old.value)
