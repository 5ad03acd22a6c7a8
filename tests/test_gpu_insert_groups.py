"""Inserts whose groups hold eight edges each (one wave per CU, batches of some
15,000 edges and up; at the default a group has one edge until 65,536, eight
past 458,752), against the oracle's CSR: one bucket a group, buckets shared by
some, chains that fill within a group, duplicates, tombstones."""
import ctypes

import numpy as np
import pytest
from test_gpu_insert_paths import check

import meerkat_amd as mk
from meerkat_amd import _lib, gen

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def one_wave_per_cu(gpu):
    old = ctypes.c_int64()
    _lib.call("mk_tune_get", b"mut_waves_per_cu", ctypes.byref(old))
    _lib.call("mk_tune_set", b"mut_waves_per_cu", 1)
    yield
    _lib.call("mk_tune_set", b"mut_waves_per_cu", old.value)


def insert(g, s, d, w):
    """Insert, and check the statuses against the graph's keys so far."""
    before = gen.keys_of(*mk_edges(g)) if g.num_edges() else np.zeros(0, np.uint64)
    g.InsertEdges(s, d, w)
    st, keys, loop = g.last_status(), gen.keys_of(s, d), s == d
    assert (st[loop] == 2).all() and np.isin(st[~loop], (0, 1)).all()
    new = np.setdiff1d(keys[~loop], before)
    assert np.array_equal(np.sort(keys[st == 1]), new)  # each new key once


def mk_edges(g):
    row, col, _ = g.export_csr()
    return np.repeat(np.arange(g.n, dtype=np.uint32), np.diff(row).astype(int)), col


def weights_of(keys):
    return ((keys * np.uint64(2654435761)) >> np.uint64(20)).astype(np.uint32) | np.uint32(1)


# csz = ceil(ceil(count / 256 waves) / 8): eight from 14,337 on (256 CUs);
# remainders of 8 and of 64 behind
@pytest.mark.parametrize("count", [14_337, 14_344, 16_384, 16_385, 16_391, 16_447, 20_003])
@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("kind", ["runs", "mixed", "one", "repeated"])
def test_groups_of_eight(gpu, count, weighted, kind):
    n = 1 << 15
    rng = np.random.default_rng(count)
    at = np.arange(count)
    if kind == "runs":      # eight edges a source and a bucket
        s, d = at // 8, rng.integers(0, n, count)
    elif kind == "mixed":   # two of eight share a bucket, six have their own
        s = np.where(at % 8 < 2, at // 8, n // 2 + at % (n // 2))
        d = rng.integers(0, n, count)
    elif kind == "one":     # every edge in the chains of four buckets
        s, d = at * 4 // count, rng.permutation(n)[:count]
    else:                   # pairs and fours of one key, self-loops between
        s = at // 8
        d = rng.integers(0, n, count)[at // np.where(at % 16 < 8, 2, 4) * 2 % count]
        d = np.where(at % 11 == 3, s, d)
    s, d = s.astype(np.uint32), d.astype(np.uint32)
    keys = gen.keys_of(s, d)
    w = weights_of(keys) if weighted else None
    pool = mk.SlabPool(1 << 25)
    g = mk.DynamicGraph(n, pool, 0.7, None, weighted=weighted, reverse=True)
    insert(g, s, d, w)
    want = np.unique(keys[s != d])
    check(g, want, weights_of(want) if weighted else None)
    # a third deleted, then everything offered again in reverse order
    gone = want[::3]
    g.DeleteEdges(*gen.split_keys(gone))
    left = np.setdiff1d(want, gone)
    check(g, left, weights_of(left) if weighted else None)
    insert(g, s[::-1].copy(), d[::-1].copy(), None if w is None else w[::-1].copy())
    check(g, want, weights_of(want) if weighted else None)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("order", ["sorted", "shuffled"])
@pytest.mark.parametrize("load", [0.7, 4.0])
def test_rmat_in_eights(gpu, weighted, order, load):
    n, s, d, w = gen.rmat(13, 16, seed=22, weighted=True)
    keys = gen.keys_of(s, d)
    at = np.arange(len(s)) if order == "sorted" else np.random.default_rng(2).permutation(len(s))
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, load, gen.degree_hints(n, s), weighted=weighted, reverse=True,
                        in_degree_hints=gen.degree_hints(n, d))
    insert(g, s[at], d[at], w[at] if weighted else None)
    check(g, keys, w if weighted else None)
