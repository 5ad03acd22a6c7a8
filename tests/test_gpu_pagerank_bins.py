"""PageRank iterations over the packed in-adjacency against the oracle's FP64
PageRank, at the edges of the bins and of the source parts.

Tolerance: L1 <= 1e-6 against the ranks at delta 1e-14, for a stop at L1
delta 1e-7: the tail after stopping is at most d / (1 - d) * 1e-7 = 5.7e-7,
and n float32 ranks that sum to 1 are within 6e-8 of it in rounding.
"""
import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


def reference(n, s, d):
    g = oracle.csr(n, s, d)
    pr, _, delta = oracle.pagerank(oracle.transpose(g), g.degrees(), 0.85, 1e-14, 5000)
    assert delta <= 1e-14
    return pr


def edges(n, scale, seed):
    """RMAT edges on the first 2**scale ids (hubs: bins split into items)
    with uniform edges over all n, the last vertex among them."""
    _, s, d, _ = gen.rmat(scale, 8, seed=seed)
    us, ud, _ = gen.insert_batch(None, n, 2 * n, seed=seed + 1)
    keys = np.unique(np.r_[gen.keys_of(s, d), gen.keys_of(us, ud),
                           gen.keys_of(np.uint32([n - 1]), np.uint32([0])),
                           gen.keys_of(np.uint32([3]), np.uint32([n - 1]))])
    return gen.split_keys(keys[(keys >> np.uint64(32)) != (keys & np.uint64(0xFFFFFFFF))])


@pytest.mark.parametrize("n,scale,weighted,hints", [
    (256, 7, False, True),         # one bin
    (257, 8, True, False),         # the second bin holds one vertex
    (131072, 15, False, False),    # one source part; long chains
    (131073, 16, True, True),      # bins of 2^9; the second part holds one vertex
    (524288 + 77, 19, False, True),  # bins of 2^11, split ones among them
    (600011, 17, True, False),
])
@pytest.mark.parametrize("mirror", [False, True])
def test_packed_iterations(gpu, n, scale, weighted, hints, mirror):
    s, d = edges(n, scale, seed=n % 1000 + scale)
    w = np.ones(len(s), np.uint32) if weighted else None
    pool = mk.SlabPool(1 << 29)
    ho, hi = (gen.degree_hints(n, s), gen.degree_hints(n, d)) if hints else (None, None)
    if mirror:
        g = mk.DynamicGraph(n, pool, 0.7, ho, weighted=weighted, reverse=True, in_degree_hints=hi)
        g.InsertEdges(s, d, w)
        pr = mk.PageRank(g, 0.85, 1e-7)
    else:
        g = mk.DynamicGraph(n, pool, 0.7, hi, weighted=weighted)
        g.InsertEdges(d, s, w)
        pr = mk.PageRank(g, 0.85, 1e-7, out_degree=gen.degree_hints(n, s))

    def check():
        v = pr.Values().astype(np.float64)
        assert np.isfinite(v).all()
        err = float(np.abs(v - reference(n, s, d)).sum())
        assert err <= 1e-6, err
        assert pr.last_stats()["iterations"] > 2

    pr.Static()
    check()
    # tombstones, then more edges than before (the packed words grow)
    keys = gen.keys_of(s, d)
    ds, dd = gen.delete_batch(keys, len(keys) // 5, seed=5)
    g.DeleteEdges(*((ds, dd) if mirror else (dd, ds)))
    pr.Decremental(ds, dd)
    keys = keys[~np.isin(keys, gen.keys_of(ds, dd))]
    s, d = gen.split_keys(keys)
    check()
    bs, bd, _ = gen.insert_batch(keys, n, len(keys) // 2, seed=6)
    bw = np.ones(len(bs), np.uint32) if weighted else None
    g.InsertEdges(*((bs, bd, bw) if mirror else (bd, bs, bw)))
    pr.Incremental(bs, bd)
    s, d = np.r_[s, bs], np.r_[d, bd]
    check()
