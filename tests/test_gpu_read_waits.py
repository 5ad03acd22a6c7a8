"""A result read behind work that is still queued: it waits without holding up
reads of other handles, and without keeping processors busy."""
import threading
import time

import numpy as np
import pytest

import meerkat_amd as mk
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


def test_read_behind_a_long_queue(gpu):
    # 64 sources in a corner of a grid of 4.2M vertices (16 chunks a result):
    # thousands of steps, queued in a fraction of the time they take
    k = 2048
    n = k * k
    i = np.arange(n, dtype=np.uint32)
    r, b = i[i % k != k - 1], i[:k * (k - 1)]
    s, d = np.r_[r, r + 1, b, b + k], np.r_[r + 1, r, b + k, b]
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, s), weighted=True)
    g.InsertEdges(s, d, (i[s] % 7 + 1).astype(np.uint32))
    other = mk.DynamicGraph(1 << 20, pool, 0.7, None)
    other.InsertEdges(np.uint32([4]), np.uint32([3]))
    # (streams share hardware queues: some of these may be behind the steps)
    ccs = [mk.CC(other) for _ in range(3)]
    labels = np.arange(1 << 20, dtype=np.uint32)
    labels[4] = 3
    for cc in ccs:
        cc.Static()
        assert np.array_equal(cc.Labels(), labels)
    q = mk.MultiSource(g, sssp=True)
    q.run([0])  # the stage and the handle's arrays are there
    first = q.distances(0)
    q.open()
    q.admit(list(range(64)), list(range(64)))
    got, ended, right = [], [], []

    def behind():
        got.append(q.distances(0))
        ended.append(time.perf_counter())

    def beside(cc):
        right.append(np.array_equal(cc.Labels(), labels))
        ended.append(time.perf_counter())

    waited = threading.Thread(target=behind)
    others = [threading.Thread(target=beside, args=(cc,)) for cc in ccs]
    q.launch(3500)
    assert not q.ready()
    wall, cpu = time.perf_counter(), time.process_time()
    waited.start()
    time.sleep(0.005)
    for t in others:
        t.start()
    for t in [waited] + others:
        t.join()
    took, cpu = [t - wall for t in ended], time.process_time() - cpu
    wall = time.perf_counter() - wall
    assert right == [True] * 3
    assert wall > 0.05 and min(took) < wall / 2, (wall, took)
    # the waiting threads may poll; those that copy have nothing to do
    assert cpu < 6 * wall, (wall, cpu)
    while q.poll()[0]:
        q.launch(64)
    assert np.array_equal(q.distances(0), first) and len(got[0]) == n
