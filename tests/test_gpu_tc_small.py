"""Static triangle counts whose list lengths the host does not wait for (up to
256 vertices, or 65,536 stored edges): closed forms and the oracle at both
edges of that range, and one-directional graphs against the same count with
every length waited for (a bound on the scratch selects that)."""
import ctypes

import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import _lib, gen

pytestmark = pytest.mark.gpu


def graph(n, s, d, weighted=False):
    pool = mk.SlabPool(1 << 24)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s), weighted=weighted)
    if len(s):
        g.InsertEdges(s, d, np.ones(len(s), np.uint32) if weighted else None)
    return g


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("n", [1, 2, 3, 65, 255, 256, 257, 1000])
def test_cliques(gpu, n, weighted):
    k = min(n, 257)  # 257 * 256 stored edges are past the range, 256 * 255 in it
    a, b = np.divmod(np.arange(k * k, dtype=np.uint32), np.uint32(k))
    m = a != b
    tc = mk.TC(graph(n, a[m], b[m], weighted))
    for _ in range(2):
        tc.Static()
        assert tc.GetCount() == k * (k - 1) * (k - 2) // 6


@pytest.mark.parametrize("n", [256, 300, 5000])
@pytest.mark.parametrize("stored", [0, 2, 64, 65_534, 65_536, 65_538])
def test_stored_edges_around_the_limit(gpu, n, stored):
    a, b = np.triu_indices(n, 1)
    stored = min(stored, 2 * len(a))
    at = np.random.default_rng(stored + n).choice(len(a), stored // 2, replace=False)
    a, b = a[at].astype(np.uint32), b[at].astype(np.uint32)
    s, d = np.r_[a, b], np.r_[b, a]
    tc = mk.TC(graph(n, s, d))
    tc.Static()
    assert tc.GetCount() == (oracle.tc(oracle.csr(n, s, d)) if stored else 0)


@pytest.mark.parametrize("n,m", [(200, 8000), (256, 32_640), (3000, 60_000)])
def test_one_direction(gpu, n, m):
    a, b = np.triu_indices(n, 1)
    at = np.random.default_rng(m).choice(len(a), min(m, len(a)), replace=False)
    tc = mk.TC(graph(n, a[at].astype(np.uint32), b[at].astype(np.uint32)))
    tc.Static()
    first = tc.GetCount()
    old = ctypes.c_int64()
    _lib.call("mk_tune_get", b"tc_scratch_mb", ctypes.byref(old))
    try:
        _lib.call("mk_tune_set", b"tc_scratch_mb", 512)
        tc.Static()
        assert tc.GetCount() == first
    finally:
        _lib.call("mk_tune_set", b"tc_scratch_mb", old.value)
