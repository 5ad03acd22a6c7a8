"""Results read to host memory in chunks of 2^18 words: sizes at the chunk,
block and slot edges, unaligned destinations, a null output, and readers on
several threads."""
import ctypes
import threading

import numpy as np
import pytest

import meerkat_amd as mk
from meerkat_amd import _lib

pytestmark = pytest.mark.gpu
CHUNK = 1 << 18


def star(n, weighted=False):
    """0 -> every 7th vertex; distances 0, 1 or unreachable."""
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, None, weighted=weighted)
    d = np.arange(7, n, 7, dtype=np.uint32)
    if len(d):
        g.InsertEdges(np.zeros(len(d), np.uint32), d, np.full(len(d), 5, np.uint32))
    want = np.full(n, mk.INF, np.uint32)
    want[0] = 0
    want[d] = 5 if weighted else 1
    return g, want


@pytest.mark.parametrize("n", [1, 2, 63, 65535, CHUNK - 1, CHUNK, CHUNK + 1, 3 * CHUNK + 5,
                               9 * CHUNK + 7])
def test_distances_parents_labels(gpu, n):
    g, want = star(n)
    b = mk.BFS(g, 0)
    b.Static()
    assert np.array_equal(b.Distances(), want)
    d, p = b.read()
    assert np.array_equal(d, want)
    reached = np.flatnonzero(want == 1)
    assert (p[reached] == 0).all() and np.array_equal(b.Parents()[reached], p[reached])
    cc = mk.CC(g)
    cc.Static()
    lab = np.arange(n, dtype=np.uint32)
    lab[reached] = 0
    assert np.array_equal(cc.Labels(), lab)
    assert np.array_equal(g.degrees(), np.r_[len(reached), np.zeros(n - 1)])


def test_unaligned_and_null_outputs(gpu):
    n = CHUNK + 3
    g, want = star(n, weighted=True)
    s = mk.SSSP(g, 0)
    s.Static()
    raw = np.zeros(4 * n + 64, np.uint8)
    out = raw[3:3 + 4 * n]
    _lib.call("mk_sssp_read", s.handle, out.ctypes.data_as(ctypes.c_void_p), None)
    assert np.array_equal(np.frombuffer(out.tobytes(), np.uint32), want)
    assert not raw[:3].any() and not raw[3 + 4 * n:].any()
    _lib.call("mk_sssp_read", s.handle, None, None)
    m = mk.MultiSource(g, sssp=True)
    m.run([0, 7, 0])
    assert np.array_equal(m.distances(2), want)
    one = np.full(n, mk.INF, np.uint32)
    one[7] = 0
    assert np.array_equal(m.distances(1), one)


def test_readers_on_several_threads(gpu):
    made = [star(2 * CHUNK + 11 + i) for i in range(3)]
    bad = []

    def reader(g, want):
        lab = np.arange(g.n, dtype=np.uint32)
        lab[want == 1] = 0
        cc = mk.CC(g)
        for _ in range(5):
            cc.Static()
            if not np.array_equal(cc.Labels(), lab):
                bad.append(g.n)
        cc.close()

    ts = [threading.Thread(target=reader, args=m) for m in made]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
