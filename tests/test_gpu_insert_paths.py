"""Inserts whose groups of eight edges share buckets, and those whose edges
all have their own, against the oracle's CSR (keys, kept weights, degrees,
statuses): sorted, shuffled and adversarial orders, duplicates within a
group, full chains, tombstones with old weights."""
import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


def check(g, keys, w):
    s, d = gen.split_keys(keys)
    ref = oracle.csr(g.n, s, d, w)
    row, col, ww = g.export_csr()
    assert np.array_equal(row, ref.row_off) and np.array_equal(col, ref.col)
    if w is not None:
        assert np.array_equal(ww, ref.w)
    assert np.array_equal(g.degrees(), np.bincount(s, minlength=g.n).astype(np.uint32))
    if g.reverse:
        rs, rd = d, s
        order = np.lexsort((rd, rs))
        row, col, ww = g.mirror().export_csr()
        assert np.array_equal(col, rd[order])
        if w is not None:
            assert np.array_equal(ww, w[order])


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("order", ["sorted", "shuffled", "by-dst"])
@pytest.mark.parametrize("hints", [True, False])
def test_orders(gpu, weighted, order, hints):
    n, s, d, w = gen.rmat(13, 16, seed=21, weighted=True)
    keys = gen.keys_of(s, d)
    at = {"sorted": np.arange(len(s)), "by-dst": np.lexsort((s, d)),
          "shuffled": np.random.default_rng(1).permutation(len(s))}[order]
    pool = mk.SlabPool(1 << 26)
    h = gen.degree_hints(n, s) if hints else None
    hi = gen.degree_hints(n, d) if hints else None
    g = mk.DynamicGraph(n, pool, 0.7, h, weighted=weighted, reverse=True, in_degree_hints=hi)
    g.InsertEdges(s[at], d[at], w[at] if weighted else None)
    assert (g.last_status() == 1).all()
    check(g, keys, w if weighted else None)
    # half deleted, put back with other weights over their tombstones
    gone = np.arange(0, len(s), 2)
    g.DeleteEdges(s[gone], d[gone])
    w = w.copy()
    w[gone] += 1000
    back = at[np.isin(at, gone)]
    g.InsertEdges(s[back], d[back], w[back] if weighted else None)
    assert (g.last_status() == 1).all()
    check(g, keys, w if weighted else None)
    # all again: present, weights kept
    g.InsertEdges(s[at], d[at], (w[at] + 7) if weighted else None)
    assert (g.last_status() == 0).all()
    check(g, keys, w if weighted else None)


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("count", [1, 7, 8, 9, 63, 64, 65, 70000])
def test_duplicates_in_a_group(gpu, weighted, count):
    # each edge eight times in a row, self-loops between; every size around
    # a group and a wave
    n = 4096
    rng = np.random.default_rng(count)
    s = np.repeat(rng.integers(0, 64, count), 8)[:count].astype(np.uint32)
    d = np.repeat(rng.integers(0, n, count), 8)[:count].astype(np.uint32)
    d[::5] = s[::5]
    w = np.full(count, 9, np.uint32) if weighted else None
    pool = mk.SlabPool(1 << 24)
    g = mk.DynamicGraph(n, pool, 0.7, None, weighted=weighted, reverse=True)
    g.InsertEdges(s, d, w)
    st = g.last_status()
    loop = s == d
    assert (st[loop] == 2).all() and np.isin(st[~loop], (0, 1)).all()
    keys = np.unique(gen.keys_of(s, d)[~loop])
    assert int((st == 1).sum()) == len(keys)
    check(g, keys, np.full(len(keys), 9, np.uint32) if weighted else None)
