"""Components of graphs that the sampling steps join slowly (uniform graphs of
every density, permuted paths and grids, cliques in a ring, trees): labels
against the oracle, sets and maps, edges held in one or both directions."""
import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


def shape(name, rng):
    if name.startswith("er"):
        n, m = (int(x) for x in name[2:].split("x"))
        s, d, _ = gen.insert_batch(None, n, m, seed=m)
        return n, s, d
    if name == "path":
        q = rng.permutation(70_001)
        return 70_001, q[:-1], q[1:]
    if name == "grid":
        k = 200
        i, q = np.arange(k * k), rng.permutation(k * k)
        r, b = i[i % k != k - 1], i[:k * (k - 1)]
        return k * k, q[np.r_[r, b]], q[np.r_[r + 1, b + k]]
    if name == "tree":
        n = 50_000
        return n, np.arange(1, n), (rng.random(n - 1) * np.arange(1, n)).astype(int)
    k, c = 90, 40  # cliques, joined in a ring but for one gap
    x, y = np.triu_indices(k, 1)
    at = k * np.arange(c)[:, None]
    return k * c, np.r_[(x + at).ravel(), k * np.arange(c - 1)], \
        np.r_[(y + at).ravel(), k * np.arange(1, c)]


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("both", [False, True])
@pytest.mark.parametrize("name", ["er65x40", "er20000x10000", "er20000x40000", "er20000x320000",
                                  "er131072x1048576", "path", "grid", "tree", "cliques"])
def test_labels(gpu, name, both, weighted):
    n, s, d = shape(name, np.random.default_rng(len(name)))
    s, d = s.astype(np.uint32), d.astype(np.uint32)
    two = np.unique(np.r_[gen.keys_of(s, d), gen.keys_of(d, s)])
    want = oracle.cc(oracle.csr(n, *gen.split_keys(two)))[0]
    if both:
        s, d = gen.split_keys(two)
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s), weighted=weighted)
    g.InsertEdges(s, d, np.ones(len(s), np.uint32) if weighted else None)
    cc = mk.CC(g)
    for _ in range(2):
        cc.Static()
        assert np.array_equal(cc.Labels(), want)
