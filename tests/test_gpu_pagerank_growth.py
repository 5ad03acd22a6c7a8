"""PageRank over packed words whose number grows, call by call, to the end of
the room kept to spare and past it, against the oracle's FP64 PageRank.

Tolerance as for the other packed iterations: L1 <= 1e-6 against the ranks at
delta 1e-14, for a stop at L1 delta 1e-7 (5.7e-7 of tail, 6e-8 of rounding).
"""
import numpy as np
import pytest

import meerkat_amd as mk
import oracle
from meerkat_amd import gen, profiling

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [4001, 4002, 4007])
def test_words_at_the_end_of_their_buffer(gpu, first):
    n = 700
    room = first + first // 8 + 64
    s, d, _ = gen.insert_batch(None, n, room + 2, seed=first)
    pool = mk.SlabPool(1 << 24)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s), reverse=True)
    g.InsertEdges(s[:first], d[:first])
    pr = mk.PageRank(g, 0.85, 1e-7)
    pr.Static()
    at = first
    for upto in (room - 5, room - 3, room - 2, room - 1, room, room + 1, room + 2):
        bs, bd = mk.device_u32(s[at:upto]), mk.device_u32(d[at:upto])
        g.InsertEdges(bs, bd)
        pr.Incremental(bs, bd)
        at = upto
        ref = oracle.csr(n, s[:at], d[:at])
        want, _, delta = oracle.pagerank(oracle.transpose(ref), ref.degrees(), 0.85, 1e-14, 5000)
        assert delta <= 1e-14 and pr.last_stats()["iterations"] > 2
        assert np.abs(pr.Values().astype(np.float64) - want).sum() <= 1e-6


def test_call_of_one_iteration_launches_one(gpu):
    # ranks that still hold: the call ends with the wait after its first
    # iteration
    n, s, d, _ = gen.rmat(12, 8, seed=6)
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s), reverse=True)
    g.InsertEdges(s, d)
    pr = mk.PageRank(g, 0.85, 1e-6)
    pr.Static()
    many = pr.last_stats()["iterations"]
    ranks = pr.Values()
    profiling.enable()
    try:
        profiling.reset()
        pr.Static()
        used = profiling.totals()
    finally:
        profiling.enable(False)
    assert many > 2 and pr.last_stats()["iterations"] == 1
    assert used["k_pr_iterate"]["launches"] == 1
    assert np.abs(pr.Values().astype(np.float64) - ranks).sum() <= 1e-6


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("n,degree", [(600, 500), (3001, 400), (16_385, 250), (9000, 700)])
def test_small_bins(gpu, n, degree, weighted):
    # many edges a vertex: bins of 32 to 128 vertices, the last not full
    s, d, _ = gen.insert_batch(None, n, n * degree, seed=n)
    hub = np.arange(1, n, dtype=np.uint32)  # one vertex that all others name
    keys = np.unique(np.r_[gen.keys_of(s, d), gen.keys_of(hub, np.zeros(n - 1, np.uint32))])
    s, d = gen.split_keys(keys)
    pool = mk.SlabPool(1 << 28)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s), weighted=weighted, reverse=True,
                        in_degree_hints=gen.degree_hints(n, d))
    g.InsertEdges(s, d, np.ones(len(s), np.uint32) if weighted else None)
    pr = mk.PageRank(g, 0.85, 1e-7)
    pr.Static()
    ref = oracle.csr(n, s, d)
    want, _, delta = oracle.pagerank(oracle.transpose(ref), ref.degrees(), 0.85, 1e-14, 5000)
    assert delta <= 1e-14 and pr.last_stats()["iterations"] > 2
    assert np.abs(pr.Values().astype(np.float64) - want).sum() <= 1e-6
