"""Multi-source SSSP steps that go over all buckets (wide frontiers) and the
changes between them and queued steps, against the oracle's Dijkstra
(bit-exact): few and many sources, chains of several slabs, tiny graphs,
sources admitted while a scan's frontier has no queue, weights near the top
of 32 bits."""
import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import gen
from test_gpu_sessions import run_session

pytestmark = pytest.mark.gpu


def graph(n, s, d, w, hints=True):
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s) if hints else None, weighted=True)
    g.InsertEdges(s, d, w)
    return g, oracle.csr(n, s, d, w)


@pytest.mark.parametrize("hints", [True, False])
@pytest.mark.parametrize("scale, k", [(1, 1), (4, 3), (8, 4), (11, 5), (13, 33), (13, 64)])
def test_runs(gpu, scale, k, hints):
    n, s, d, w = gen.rmat(scale, 8, seed=scale + k, weighted=True)
    g, ref = graph(n, s, d, w, hints)
    q = mk.MultiSource(g, sssp=True)
    for seed in range(2):
        srcs = np.random.default_rng(seed).integers(0, n, k).astype(np.uint32)
        q.run(srcs)
        for slot, v in enumerate(srcs):
            assert np.array_equal(q.distances(slot), oracle.dijkstra(ref, int(v))), slot


@pytest.mark.parametrize("n", [63, 64, 65, 2047, 2048, 2049])
def test_wide_then_narrow_then_wide(gpu, n):
    # a star into every vertex, a path out of one of them, a second star at
    # its end that improves every vertex again
    path = 20
    a = np.arange(1, n - path - 1, dtype=np.uint32)
    p = np.arange(n - path - 1, n - 1, dtype=np.uint32)
    s = np.r_[np.zeros(len(a), np.uint32), a[0], p[:-1], p[-1], np.full(len(a) - 1, n - 1, np.uint32)]
    d = np.r_[a, p[0], p[1:], n - 1, a[1:]]
    w = np.r_[np.full(len(a), 1000, np.uint32), np.ones(path + 1, np.uint32),
              np.arange(1, len(a), dtype=np.uint32)].astype(np.uint32)
    w[0] = 1
    g, ref = graph(n, s.astype(np.uint32), d.astype(np.uint32), w)
    q = mk.MultiSource(g, sssp=True)
    srcs = np.r_[np.zeros(6, np.uint32), n - 1, a[0], p].astype(np.uint32)[:40]
    q.run(srcs)
    for slot, v in enumerate(srcs):
        assert np.array_equal(q.distances(slot), oracle.dijkstra(ref, int(v))), slot


@pytest.mark.parametrize("top", [2**31, 2**32 - 1])
def test_sums_past_32_bits_stay_unreached(gpu, top):
    # 0 -> 1 -> {2..}: the second hop overflows for the largest weights
    n = 512
    d = np.arange(2, n, dtype=np.uint32)
    s = np.r_[np.zeros(1, np.uint32), np.ones(len(d), np.uint32)]
    w = np.r_[np.uint32(2**31), np.where(d % 2, top, 5)].astype(np.uint32)
    pool = mk.SlabPool(1 << 22)
    g = mk.DynamicGraph(n, pool, 0.7, None, weighted=True)
    g.InsertEdges(s, np.r_[np.uint32(1), d].astype(np.uint32), w)
    q = mk.MultiSource(g, sssp=True)
    q.run(np.r_[np.zeros(5), 1].astype(np.uint32))
    exp = np.full(n, mk.INF, np.uint64)
    exp[0], exp[1] = 0, 2**31
    sums = 2**31 + w[1:].astype(np.uint64)
    exp[2:] = np.where(sums < mk.INF, sums, mk.INF)
    for slot in range(5):
        assert np.array_equal(q.distances(slot), exp.astype(np.uint32)), slot


@pytest.mark.parametrize("gap", [1, 2, 3])
def test_sources_admitted_between_scans(gpu, gap):
    n, s, d, w = gen.rmat(12, 16, seed=9, weighted=True)
    g, ref = graph(n, s, d, w)
    srcs = np.random.default_rng(gap).integers(0, n, 48).astype(np.uint32)
    q = mk.MultiSource(g, sssp=True)
    waves = []
    for i in range(0, 48, 8):
        waves.append([(i + j, int(v)) for j, v in enumerate(srcs[i:i + 8])])
        waves.extend([] for _ in range(gap - 1))
    run_session(q, waves)
    for slot, v in enumerate(srcs):
        assert np.array_equal(q.distances(slot), oracle.dijkstra(ref, int(v))), slot
