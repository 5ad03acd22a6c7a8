"""Traversals over long slab chains (no degree hints: one bucket a vertex), one
or several of them in a wave: static, after deletions and insertions, against
the oracle; sets and maps, with the in-edge mirror and without."""
import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


def hubs(n, count, degree, seed):
    """`count` vertices next to each other with `degree` edges each, both
    ways, over a sparse uniform graph."""
    rng = np.random.default_rng(seed)
    h = np.repeat(100 + np.arange(count), degree)
    o = np.concatenate([rng.choice(n, degree, replace=False) for _ in range(count)])
    s, d, _ = gen.insert_batch(None, n, n, seed=seed)
    keys = np.r_[gen.keys_of(s, d), gen.keys_of(h.astype(np.uint32), o.astype(np.uint32)),
                 gen.keys_of(o.astype(np.uint32), h.astype(np.uint32))]
    keys = np.unique(keys)
    return keys[(keys >> np.uint64(32)) != (keys & np.uint64(0xFFFFFFFF))]


def check(alg, keys, n, w, weights):
    s, d = gen.split_keys(keys)
    ref = oracle.csr(n, s, d, w)
    dist, par = alg.read()
    want = oracle.dijkstra(ref, alg.source) if weights else oracle.bfs(ref, alg.source)
    assert np.array_equal(dist, want)
    assert oracle.check_parents_fast(ref, dist, par, alg.source, weights=weights) == 0


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("mirror", [False, True])
@pytest.mark.parametrize("count,degree", [(1, 3000), (2, 2000), (3, 700), (9, 500), (40, 130)])
def test_hub_chains(gpu, weighted, mirror, count, degree):
    n = 6000
    keys = hubs(n, count, degree, seed=count)
    s, d = gen.split_keys(keys)
    w = (np.random.default_rng(7).integers(1, 50, len(keys)).astype(np.uint32)
         if weighted else None)
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, None, weighted=weighted, reverse=mirror)
    g.InsertEdges(s, d, w)
    algs = [mk.BFS(g, 5)] + ([mk.SSSP(g, 5)] if weighted else [])
    for a in algs:
        a.Static()
        check(a, keys, n, w, isinstance(a, mk.SSSP))
    gone = np.sort(np.random.default_rng(8).choice(len(keys), len(keys) // 4, replace=False))
    ds, dd = mk.device_u32(s[gone]), mk.device_u32(d[gone])
    dw = mk.device_u32(w[gone]) if weighted else None
    keep = np.setdiff1d(np.arange(len(keys)), gone)
    g.DeleteEdges(ds, dd)
    for a in algs:
        a.Decremental(ds, dd)
        check(a, keys[keep], n, w[keep] if weighted else None, isinstance(a, mk.SSSP))
    g.InsertEdges(ds, dd, dw)
    for a in algs:
        a.Incremental(ds, dd)
        check(a, keys, n, w, isinstance(a, mk.SSSP))
