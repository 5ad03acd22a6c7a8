"""Static traversals whose frontiers are large enough for dense steps, against
the oracle (distances bit-exact, parents valid): distances below, at and past
what a 16-bit bound holds, chained slabs, tombstones, set and map slabs, then
updates on top."""
import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


def check(g, alg, keys, n, w, source, weights):
    s, d = gen.split_keys(keys)
    ref = oracle.csr(n, s, d, w)
    dist, par = alg.read()
    want = oracle.dijkstra(ref, source) if weights else oracle.bfs(ref, source)
    assert np.array_equal(dist, want)
    assert oracle.check_parents_fast(ref, dist, par, source, weights=weights) == 0


@pytest.mark.parametrize("lo,hi,lf", [
    (1, 100, 0.7), (0, 3, 4.0), (65533, 65537, 0.7), (1, 1 << 20, 0.7), (1 << 27, 1 << 28, 0.7),
])
def test_sssp_weights(gpu, lo, hi, lf):
    n, s, d, _ = gen.rmat(18, 16, seed=31, weighted=False)
    w = np.random.default_rng(lo + hi).integers(lo, hi, len(s)).astype(np.uint32)
    keys = gen.keys_of(s, d)
    pool = mk.SlabPool(1 << 29)
    g = mk.DynamicGraph(n, pool, lf, gen.degree_hints(n, s), weighted=True)
    g.InsertEdges(s, d, w)
    src = int(s[len(s) // 2])
    sp = mk.SSSP(g, src)
    for _ in range(2):  # the second run over the first one's state
        sp.Static()
        check(g, sp, keys, n, w, src, True)
    ds, dd = gen.delete_batch(keys, len(keys) // 4, seed=3)
    g.DeleteEdges(ds, dd)
    keep = ~np.isin(keys, gen.keys_of(ds, dd))
    keys, w = keys[keep], w[keep]
    sp.Decremental(ds, dd)
    check(g, sp, keys, n, w, src, True)
    sp.set_source(0)
    sp.Static()  # over tombstones
    check(g, sp, keys, n, w, 0, True)


@pytest.mark.parametrize("weighted,lf", [(False, 0.7), (True, 0.7), (False, 8.0)])
def test_bfs_without_mirror(gpu, weighted, lf):
    # more than 2^19 buckets; RMAT hubs over uniform edges
    n = (1 << 20) + 5
    _, s, d, _ = gen.rmat(19, 8, seed=5)
    us, ud, _ = gen.insert_batch(None, n, 2 * n, seed=6)
    keys = np.unique(np.r_[gen.keys_of(s, d), gen.keys_of(us, ud)])
    s, d = gen.split_keys(keys)
    keys = keys[s != d]
    s, d = gen.split_keys(keys)
    pool = mk.SlabPool(1 << 30)
    g = mk.DynamicGraph(n, pool, lf, gen.degree_hints(n, s), weighted=weighted)
    g.InsertEdges(s, d, np.ones(len(s), np.uint32) if weighted else None)
    b = mk.BFS(g, n - 1)
    for src in (n - 1, 0):
        b.set_source(src)
        b.Static()
        check(g, b, keys, n, None, src, False)
    bs, bd, bw = gen.insert_batch(keys, n, 50000, seed=8, weighted=True)
    g.InsertEdges(bs, bd, bw if weighted else None)
    b.Incremental(bs, bd)
    check(g, b, np.sort(np.r_[keys, gen.keys_of(bs, bd)]), n, None, 0, False)
