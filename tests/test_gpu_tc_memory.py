"""Device memory of triangle counting: batches whose edges' buckets are more
than the bound on work items (worked in windows, the count exact)."""
import numpy as np
import pytest
import torch

import meerkat_amd as mk
from meerkat_amd import gen

pytestmark = pytest.mark.gpu


def held(call):
    """Bytes of device memory that `call` leaves allocated."""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    call()
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("weighted,hubs,share", [(False, 300, 0.325), (True, 200, 0.4)])
def test_batch_of_hub_edges(gpu, weighted, hubs, share):
    # hubs of some 13,000 / 16,000 leaves (295 / 740 buckets); the batch joins
    # all of them: 13 / 15 million (edge, bucket) pairs, against 4.2 million
    # items of 8 bytes
    leaves = 40_000
    n = hubs + leaves
    a = np.random.default_rng(hubs).random((hubs, leaves)) < share
    h, leaf = (x.astype(np.uint32) for x in np.nonzero(a))
    leaf += np.uint32(hubs)
    i, j = (x.astype(np.uint32) for x in np.nonzero(~np.eye(hubs, dtype=bool)))
    s, d = np.r_[h, leaf], np.r_[leaf, h]
    pool = mk.SlabPool(1 << 26)
    g = mk.DynamicGraph(n, pool, 0.7, gen.degree_hints(n, np.r_[s, i]), weighted=weighted)
    g.InsertEdges(s, d, np.ones(len(s), np.uint32) if weighted else None)
    tc = mk.TC(g)
    tc.Static()
    assert tc.GetCount() == 0
    common = a.astype(np.float32) @ a.T.astype(np.float32)  # whole numbers below 2^24
    want = hubs * (hubs - 1) * (hubs - 2) // 6 + int(np.triu(common, 1).astype(np.int64).sum())
    bi, bj = mk.device_u32(i), mk.device_u32(j)
    bw = mk.device_u32(np.ones(len(i), np.uint32)) if weighted else None
    for _ in range(2):
        g.InsertEdges(bi, bj, bw)
        used = held(lambda: tc.Incremental(bi, bj))
        assert tc.GetCount() == want
        assert used <= 48 << 20, used  # items 32 MB, the edges' arrays 4 MB
        g.DeleteEdges(bi, bj)
        tc.Decremental(bi, bj)
        assert tc.GetCount() == 0
