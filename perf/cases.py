"""Performance cases: the dynamic-graph work a program gives this library,
through the Python classes over the C ABI.

listed() names one case per kind of work; draw() gives further ones over the
same ranges of sizes.  Graphs are RMAT (a, b, c, d = 0.57, 0.19, 0.19, 0.05,
edge factor 16, weights 1..100, as the generators and bench.py have them) or
Erdos-Renyi (8 edges per vertex), made on the device from the seed.  A pass
that changes its graph ends with the edge set it began with, so it can be
repeated: batches are inserted and deleted again, or deleted and put back.
"""
import numpy as np
import torch

import meerkat_amd as mk

DEV = "cuda:0"
LOAD = 0.7  # the default load factor


def listed():
    return [
        # a small graph kept exact under small batches, every call waited
        # for: what an interactive user sees, launch latency throughout
        {"name": "sssp-updates-small", "kind": "updates", "algo": "sssp", "scale": 16,
         "batch": 1000, "pairs": 1, "mirror": True, "deferred": False},
        # the headline loop: large batches, in-edge mirror, deferred calls,
        # the distances read after every eight steps
        {"name": "sssp-updates-large", "kind": "updates", "algo": "sssp", "scale": 22,
         "batch": 500_000, "pairs": 8, "mirror": True, "deferred": True},
        # unweighted, no mirror (half the memory), ordinary odd-sized batches
        {"name": "bfs-updates-no-mirror", "kind": "updates", "algo": "bfs", "scale": 20,
         "batch": 20_011, "pairs": 2, "mirror": False, "deferred": False},
        # edge ingestion and lookups with no traversal attached
        {"name": "mutate-search", "kind": "mutate", "scale": 22, "batch": 999_983,
         "weighted": False, "mirror": False},
        # loading a whole weighted graph with its mirror, then dropping it
        {"name": "build", "kind": "build", "scale": 20, "weighted": True, "mirror": True},
        # one-source queries on a resident graph, distances to the host
        {"name": "bfs-static", "kind": "static", "algo": "bfs", "scale": 22, "sources": 4,
         "mirror": True},
        {"name": "sssp-static", "kind": "static", "algo": "sssp", "scale": 24, "sources": 2,
         "mirror": False},
        # ranks kept current under large batches (insert, then delete)
        {"name": "pagerank-updates", "kind": "pagerank", "graph": "er", "n": 4_194_304,
         "batch": 1_000_000, "mirror": False},
        # triangles of a social-network shaped graph, from scratch
        {"name": "triangles-static", "kind": "tc_static", "scale": 20},
        # and kept current under batches of further edges of that shape
        {"name": "triangles-updates", "kind": "tc_updates", "scale": 18, "batch": 50_021},
        # components from scratch, then kept current
        {"name": "components", "kind": "cc", "scale": 21, "batch": 200_003},
        # a full round of the serving loop: 64 queries in one traversal
        {"name": "serving-sssp-64", "kind": "multi", "algo": "sssp", "scale": 20, "sources": 64},
    ]


def _log_int(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["updates", "updates", "mutate", "build", "static", "static", "pagerank",
                       "tc_static", "tc_updates", "cc", "multi"])
    yes = lambda: rng.random() < 0.5  # noqa: E731
    if kind == "updates":
        scale = rng.randint(14, 22)
        return {"kind": kind, "algo": rng.choice(["bfs", "sssp"]), "scale": scale,
                "batch": _log_int(rng, 501, min(500_000, 1 << (scale + 1))),
                "pairs": rng.randint(1, 4), "mirror": yes(), "deferred": yes()}
    if kind == "mutate":
        scale = rng.randint(16, 22)
        return {"kind": kind, "scale": scale,
                "batch": _log_int(rng, 333, min(999_983, 1 << (scale + 2))),
                "weighted": yes(), "mirror": yes()}
    if kind == "build":
        return {"kind": kind, "scale": rng.randint(15, 20), "weighted": yes(), "mirror": yes()}
    if kind == "static":
        return {"kind": kind, "algo": rng.choice(["bfs", "sssp"]), "scale": rng.randint(16, 22),
                "sources": rng.randint(1, 4), "mirror": yes()}
    if kind == "pagerank":
        n = _log_int(rng, 100_003, 4_194_304)
        return {"kind": kind, "graph": rng.choice(["er", "rmat"]), "n": n,
                "batch": _log_int(rng, 1_001, min(n, 1_000_000)), "mirror": yes()}
    if kind == "tc_static":
        return {"kind": kind, "scale": rng.randint(15, 19)}
    if kind == "tc_updates":
        scale = rng.randint(15, 18)
        return {"kind": kind, "scale": scale, "batch": _log_int(rng, 501, 1 << (scale - 2))}
    if kind == "cc":
        scale = rng.randint(16, 21)
        return {"kind": kind, "scale": scale, "batch": _log_int(rng, 1_001, 1 << (scale - 3))}
    algo = rng.choice(["bfs", "sssp"])
    return {"kind": "multi", "algo": algo, "scale": rng.randint(15, 19),
            "sources": rng.randint(5, 64)}


# ------------------------------------------------------------------ graphs
def _rng(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _rmat_keys(n, m, gen):
    """Sorted unique src << 32 | dst of an RMAT draw of m edges over n
    vertices (ids past n, when n is no power of two, wrap), no self-loops."""
    bits = max(1, (n - 1).bit_length())
    src = torch.zeros(m, dtype=torch.int64, device=DEV)
    dst = torch.zeros(m, dtype=torch.int64, device=DEV)
    for _ in range(bits):
        r = torch.rand(m, device=DEV, generator=gen)
        hi = r >= 0.76  # lower half of the matrix: c or d
        src.mul_(2).add_(hi)
        dst.mul_(2).add_(torch.where(hi, r >= 0.95, r >= 0.57))
    if n != 1 << bits:
        src.remainder_(n)
        dst.remainder_(n)
    return torch.unique(((src << 32) | dst)[src != dst])


def _er_keys(n, m, gen):
    src = torch.randint(n, (m,), device=DEV, generator=gen)
    dst = torch.randint(n, (m,), device=DEV, generator=gen)
    return torch.unique(((src << 32) | dst)[src != dst])


def _split(keys):
    return (keys >> 32).to(torch.int32), (keys & 0xFFFFFFFF).to(torch.int32)


def _weights(count, gen):
    return torch.randint(1, 101, (count,), device=DEV, generator=gen, dtype=torch.int32)


def _degrees(n, ids):
    return torch.bincount(ids, minlength=n).to(torch.int32).cpu().numpy().view(np.uint32)


def _shuffled(count, gen):
    return torch.randperm(count, device=DEV, generator=gen)


def _new_keys(keys, n, count, gen):
    """`count` distinct uniform edges absent from `keys` (sorted), shuffled."""
    got = torch.empty(0, dtype=torch.int64, device=DEV)
    while len(got) < count:
        k = _er_keys(n, count + count // 4 + 64, gen)
        at = torch.searchsorted(keys, k).clamp_(max=len(keys) - 1)
        got = torch.unique(torch.cat([got, k[keys[at] != k]]))
    return got[_shuffled(len(got), gen)[:count]]


def _undirected(keys):
    """The edges u < v of `keys`, once each, sorted."""
    src, dst = keys >> 32, keys & 0xFFFFFFFF
    return torch.unique((torch.minimum(src, dst) << 32) | torch.maximum(src, dst))


def _both(und):
    src, dst = und >> 32, und & 0xFFFFFFFF
    return torch.cat([und, (dst << 32) | src])


def _graph(n, keys, w, mirror, pool_bytes=1 << 30):
    """The resident graph of sorted `keys`, sized from its own degrees."""
    s, d = _split(keys)
    pool = mk.SlabPool(pool_bytes)
    g = mk.DynamicGraph(n, pool, LOAD, _degrees(n, s), weighted=w is not None, reverse=mirror,
                        in_degree_hints=_degrees(n, d) if mirror else None)
    g.InsertEdges(s, d, w)
    return g


def _sources(keys, count, gen):
    """Vertices with out-edges."""
    at = torch.randint(len(keys), (count,), device=DEV, generator=gen)
    return [int(v) for v in (keys[at] >> 32).cpu()]


# ----------------------------------------------------------------- prepare
def prepare(case, seed):
    kind = case["kind"]
    gen = _rng(seed)
    if kind == "pagerank":
        return _prepare_pagerank(case, gen)
    n = 1 << case["scale"]
    keys = _rmat_keys(n, 16 * n, gen)
    if kind == "updates":
        weighted = case["algo"] == "sssp"
        w = _weights(len(keys), gen) if weighted else None
        g = _graph(n, keys, w, case["mirror"])
        alg = (mk.SSSP if weighted else mk.BFS)(g, _sources(keys, 1, gen)[0])
        alg.Static()
        pick = _shuffled(len(keys), gen)
        new = _new_keys(keys, n, case["batch"] * case["pairs"], gen)
        steps = []
        for i in range(case["pairs"]):
            at = pick[i * case["batch"]:(i + 1) * case["batch"]]
            b = new[i * case["batch"]:(i + 1) * case["batch"]]
            steps.append((_split(keys[at]) + (w[at] if weighted else None,),
                          _split(b) + (_weights(len(b), gen) if weighted else None,)))
        g.set_deferred(case["deferred"])
        alg.set_deferred(case["deferred"])
        return {"kind": kind, "alg": alg, "graph": g, "steps": steps}
    if kind == "mutate":
        w = _weights(len(keys), gen) if case["weighted"] else None
        g = _graph(n, keys, w, case["mirror"])
        at = _shuffled(len(keys), gen)[:case["batch"]]
        new = _new_keys(keys, n, case["batch"], gen)
        # lookups: a third deleted, a third added, a third untouched
        third = case["batch"] // 3
        q = torch.cat([keys[at[:third]], new[:third],
                       keys[torch.randint(len(keys), (third + 1,), device=DEV, generator=gen)]])
        q = q[_shuffled(len(q), gen)]
        return {"kind": kind, "graph": g,
                "old": _split(keys[at]) + (w[at] if w is not None else None,),
                "new": _split(new) + (_weights(len(new), gen) if w is not None else None,),
                "ask": _split(q)}
    if kind == "build":
        s, d = _split(keys)
        return {"kind": kind, "n": n, "s": s, "d": d, "mirror": case["mirror"],
                "w": _weights(len(keys), gen) if case["weighted"] else None,
                "out_hints": _degrees(n, s), "in_hints": _degrees(n, d) if case["mirror"] else None,
                "pool": mk.SlabPool(1 << 30)}
    if kind == "static":
        weighted = case["algo"] == "sssp"
        g = _graph(n, keys, _weights(len(keys), gen) if weighted else None, case["mirror"])
        src = _sources(keys, case["sources"], gen)
        return {"kind": kind, "alg": (mk.SSSP if weighted else mk.BFS)(g, src[0]), "graph": g,
                "sources": src}
    if kind == "multi":
        weighted = case["algo"] == "sssp"
        g = _graph(n, keys, _weights(len(keys), gen) if weighted else None, False)
        return {"kind": kind, "alg": mk.MultiSource(g, sssp=weighted), "graph": g,
                "sources": np.array(_sources(keys, case["sources"], gen), np.uint32)}
    # undirected graphs, both directions stored
    und = _undirected(keys)
    batch = case.get("batch", 0)
    order = _shuffled(len(und), gen)
    more = und[order[:batch]]  # held out: arrives later
    base = torch.sort(_both(und[order[batch:]]))[0]
    g = _graph(n, base, None, False)
    alg = (mk.CC if kind == "cc" else mk.TC)(g)
    if kind == "tc_updates":
        alg.Static()
    return {"kind": kind, "alg": alg, "graph": g, "more": _split(_both(more))}


def _pagerank_keys(case, gen):
    n = case["n"]
    keys = (_er_keys if case["graph"] == "er" else _rmat_keys)(n, 8 * n, gen)
    return keys, _new_keys(keys, n, case["batch"], gen)


def _prepare_pagerank(case, gen):
    n = case["n"]
    keys, new = _pagerank_keys(case, gen)
    s, d = _split(keys)
    if case["mirror"]:
        g = _graph(n, keys, None, True)
        alg = mk.PageRank(g, 0.85, 1e-7)
    else:  # a graph of the reversed edges, with the out-degrees given
        g = _graph(n, torch.sort((keys << 32) | (keys >> 32))[0], None, False)
        alg = mk.PageRank(g, 0.85, 1e-7, out_degree=_degrees(n, s))
    alg.Static()
    return {"kind": "pagerank", "alg": alg, "graph": g, "mirror": case["mirror"],
            "new": _split(new)}


# --------------------------------------------------------------------- run
def run(state):
    return _RUN[state["kind"]](state)


def _whole(a):
    """uint32 results as the int32 view of the same bits."""
    return a.view(np.int32)


def _run_updates(st):
    g, alg = st["graph"], st["alg"]
    out = []
    for back in (False, True):  # there, then back to the edges it began with
        for old, new in st["steps"]:
            gone, come = (new, old) if back else (old, new)
            g.DeleteEdges(gone[0], gone[1])
            alg.Decremental(gone[0], gone[1])
            g.InsertEdges(*come)
            if come[2] is None:
                alg.Incremental(come[0], come[1])
            else:
                alg.Incremental(*come)
        out.append(_whole(alg.Distances()))
    return out


def _run_mutate(st):
    g, old, new = st["graph"], st["old"], st["new"]
    out = []
    for gone, come in ((old, new), (new, old)):
        g.DeleteEdges(gone[0], gone[1])
        out.append(g.last_status())
        g.InsertEdges(*come)
        out.append(g.last_status())
        found = g.SearchEdges(*st["ask"])
        out += [found[0], _whole(found[1])] if isinstance(found, tuple) else [found]
    return out


def _run_build(st):
    g = mk.DynamicGraph(st["n"], st["pool"], LOAD, st["out_hints"], weighted=st["w"] is not None,
                        reverse=st["mirror"], in_degree_hints=st["in_hints"])
    g.InsertEdges(st["s"], st["d"], st["w"])
    out = [_whole(g.degrees()), g.num_edges()]
    g.close()
    return out


def _run_static(st):
    out = []
    for v in st["sources"]:
        st["alg"].set_source(v)
        st["alg"].Static()
        out.append(_whole(st["alg"].Distances()))
    return out


def _run_pagerank(st):
    g, alg, (s, d) = st["graph"], st["alg"], st["new"]
    a, b = (s, d) if st["mirror"] else (d, s)
    g.InsertEdges(a, b)
    alg.Incremental(s, d)
    up = alg.Values()
    g.DeleteEdges(a, b)
    alg.Decremental(s, d)
    return [up, alg.Values()]


def _run_tc_static(st):
    st["alg"].Static()
    return st["alg"].GetCount()


def _run_tc_updates(st):
    g, alg, (s, d) = st["graph"], st["alg"], st["more"]
    g.InsertEdges(s, d)
    alg.Incremental(s, d)
    up = alg.GetCount()
    g.DeleteEdges(s, d)
    alg.Decremental(s, d)
    return [up, alg.GetCount()]


def _run_cc(st):
    g, alg, (s, d) = st["graph"], st["alg"], st["more"]
    alg.Static()
    out = [_whole(alg.Labels())]
    g.InsertEdges(s, d)
    alg.Incremental(s, d)
    out.append(_whole(alg.Labels()))
    g.DeleteEdges(s, d)
    alg.Decremental(s, d)
    out.append(_whole(alg.Labels()))
    return out


def _run_multi(st):
    st["alg"].run(st["sources"])
    return [_whole(st["alg"].distances(i)) for i in range(len(st["sources"]))]


_RUN = {"updates": _run_updates, "mutate": _run_mutate, "build": _run_build,
        "static": _run_static, "pagerank": _run_pagerank, "tc_static": _run_tc_static,
        "tc_updates": _run_tc_updates, "cc": _run_cc, "multi": _run_multi}


# -------------------------------------------------------------------- work
def work(case):
    """Compulsory bytes and operations: batch entries, the keys (and weights)
    they name, every adjacency entry a traversal has to see once, results
    written on the device and on the host."""
    kind = case["kind"]
    if kind == "pagerank":
        n, m, b = case["n"], 8 * case["n"], case["batch"]
        # about a dozen sweeps a call (1e-7): keys, contribution in and out
        return {"bytes": 2 * (b * 12 + 12 * (4 * m + 12 * n) + 4 * n), "flops": 2 * 12 * (m + 8 * n)}
    n = 1 << case["scale"]
    m = 16 * n
    entry = 8 if case.get("algo") == "sssp" or case.get("weighted") else 4
    sides = 2 if case.get("mirror") else 1
    b = case.get("batch", 0)
    if kind == "updates":
        # per changed edge: batch entry (mutation and traversal), key word(s),
        # one distance; two reads of all distances
        edges = 4 * case["pairs"] * b
        return {"bytes": edges * (2 * (4 + entry) + sides * entry + 8) + 2 * 8 * n, "flops": edges}
    if kind == "mutate":
        return {"bytes": 6 * b * (4 + entry + sides * entry + 1), "flops": 6 * b}
    if kind == "build":
        return {"bytes": m * (4 + entry + sides * entry + 1) + 8 * n, "flops": m}
    if kind == "static":
        return {"bytes": case["sources"] * (m * entry + 12 * n), "flops": case["sources"] * m}
    if kind == "multi":
        k = case["sources"]
        return {"bytes": m * entry + k * 8 * n, "flops": k * m}
    if kind == "tc_static":
        # every edge once, and one test per wedge of the oriented graph
        # (about 150 per edge at scale 20)
        return {"bytes": 2 * m * 4 * 3, "flops": m * 150}
    if kind == "tc_updates":
        return {"bytes": 4 * b * (8 + 4) + 2 * b * 64 * 4, "flops": 2 * b * 64}
    return {"bytes": 2 * (2 * m * 4 + 8 * n) + 4 * b * 12 + 3 * 8 * n, "flops": 4 * m}


# ------------------------------------------------------------------- exact
def exact(case, seed):
    """PageRank in 64 bits with the library's stopping rule; the other kinds
    return whole numbers."""
    if case["kind"] != "pagerank":
        return None
    gen = _rng(seed)
    n = case["n"]
    keys, new = _pagerank_keys(case, gen)
    damp, margin = float(np.float32(0.85)), float(np.float32(1e-7))
    rank = torch.full((n,), 1.0 / n, dtype=torch.float64, device=DEV)

    def iterate(rank, keys):
        src, dst = keys >> 32, keys & 0xFFFFFFFF
        deg = torch.bincount(src, minlength=n).double()
        inv = torch.where(deg > 0, 1.0 / deg.clamp(min=1.0), torch.zeros_like(deg))
        for _ in range(100):
            lost = float(rank[deg == 0].sum()) / n
            acc = torch.zeros_like(rank).index_add_(0, dst, (rank * inv)[src])
            nxt = (1.0 - damp) / n + damp * acc + damp * lost
            delta = float((nxt - rank).abs().sum())
            rank = nxt
            if not delta > margin:
                break
        return rank

    rank = iterate(rank, keys)
    up = iterate(rank, torch.cat([keys, new]))
    return [up, iterate(up, keys)]
