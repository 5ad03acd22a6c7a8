"""Dense steps of static traversals at the limits of their distances: sums of
exactly 2^32 - 1 (which stands for unreached) leave a vertex without distance
and parent, and 16-bit bounds at and past their last value, improved step
after step, end in the oracle's distances."""
import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


def weighted_graph(n, s, d, w):
    order = np.lexsort((d, s))
    s, d, w = s[order], d[order], w[order]
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s), weighted=True)
    g.InsertEdges(s, d, w)
    return g, oracle.csr(n, s, d, w)


def layers(k, ways, weights):
    """A source, then layers of k vertices: vertex i of one has edges of
    weights[layer][q] to vertices i + q of the next, q < ways."""
    s, d, w = [np.zeros(k, np.uint32)], [np.arange(1, k + 1)], [np.full(k, weights[0][0])]
    for at, row in enumerate(weights[1:]):
        for q in range(ways):
            s.append(1 + at * k + np.arange(k))
            d.append(1 + (at + 1) * k + (np.arange(k) + q) % k)
            w.append(np.full(k, row[q]))
    u32 = [np.concatenate(x).astype(np.uint32) for x in (s, d, w)]
    return 1 + len(weights) * k, *u32


@pytest.mark.parametrize("first,second", [
    (5, 0xFFFFFFFF - 5), (0xFFFFFFFE, 1), (0xFFFFFFF0, 0xF), (5, 0xFFFFFFFE - 5), (5, 0xFFFFFFFF),
])
def test_sum_at_the_unreached_value(gpu, first, second):
    # a frontier of 100,000 (past a dense step's least) of some 300,000
    # buckets (past 2^18, so that the handle takes such steps)
    k = 100_000
    n, s, d, w = layers(k, 1, [[first], [second], [7]])
    g, ref = weighted_graph(n, s, d, w)
    sp = mk.SSSP(g, 0)
    for _ in range(2):
        sp.Static()
        dist, par = sp.read()
        want = np.full(n, mk.INF, np.uint64)
        want[0] = 0
        want[1:k + 1] = first
        if first + second < mk.INF:
            want[k + 1:2 * k + 1] = first + second
            if first + second + 7 < mk.INF:
                want[2 * k + 1:] = first + second + 7
        assert np.array_equal(dist, want.astype(np.uint32))
        assert (par[dist == mk.INF] == mk.INF).all()
        at = np.flatnonzero((dist != mk.INF) & (np.arange(n) > k))
        assert (par[at] == at - k).all()


@pytest.mark.parametrize("base", [65_533, 65_534, 65_535, 65_536, 1 << 20])
def test_bounds_past_16_bits(gpu, base):
    # four offers a vertex, each step's later ones better or worse by one
    n, s, d, w = layers(60_000, 4, [[base - 3], [3, 2, 1, 0], [0, 1, 2, 3], [1, 0, 1, 0],
                                    [70_000, 69_999, 1, 70_001]])
    g, ref = weighted_graph(n, s, d, w)
    sp = mk.SSSP(g, 0)
    for _ in range(2):
        sp.Static()
        dist, par = sp.read()
        assert np.array_equal(dist, oracle.dijkstra(ref, 0))
        assert oracle.check_parents_fast(ref, dist, par, 0, weights=True) == 0
