"""Re-seeding after deletions where the only path left sums to 2^32 - 1 (which
stands for unreached), past it, or to the last distance below it: with the
in-edge mirror (pull) and without (push), from one vertex to thousands,
single and hub in-neighbours."""
import numpy as np
import pytest

import meerkat_amd as mk
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mirror", [True, False])
@pytest.mark.parametrize("k", [1, 9, 5000])
@pytest.mark.parametrize("hub", [False, True])
@pytest.mark.parametrize("w", [0xE, 0xF, 0x10, 0xFFFFFFFF])
def test_remaining_path_at_the_unreached_value(gpu, mirror, k, hub, w):
    # 0 -> a_i (10) -> t_i (1); 0 -> b_i (2^32 - 16) -> t_i (w), b_0 for all
    # t_i with `hub`; every a_i -> t_i is deleted
    far = 0xFFFFFFF0
    a, b = 1 + np.arange(k), 1 + k + np.arange(k)
    t, n = 1 + 2 * k + np.arange(k), 1 + 3 * k
    from_b = np.full(k, b[0]) if hub else b
    z, one = np.zeros(k, int), np.ones(k, int)
    s = np.r_[z, z, a, from_b].astype(np.uint32)
    d = np.r_[a, b, t, t].astype(np.uint32)
    ww = np.r_[10 * one, far * one, one, w * one].astype(np.uint32)
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s), weighted=True, reverse=mirror)
    g.InsertEdges(s, d, ww)
    sp = mk.SSSP(g, 0)
    sp.Static()
    assert (sp.Distances()[t] == 11).all()
    ds, dd = a.astype(np.uint32), t.astype(np.uint32)
    g.DeleteEdges(ds, dd)
    sp.Decremental(ds, dd)
    dist, par = sp.read()
    if far + w < mk.INF:
        assert (dist[t] == far + w).all() and np.array_equal(par[t], from_b)
    else:
        assert (dist[t] == mk.INF).all() and (par[t] == mk.INF).all()
    assert (dist[a] == 10).all() and (dist[b] == far).all()
