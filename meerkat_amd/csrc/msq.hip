// Multi-source BFS / SSSP: up to 64 queries answered by one traversal.
//
// No reference counterpart (the reference runs one source per BFS/SSSP
// object, include/Algorithms/BFS.cuh:34).  Source slot s (0..63) is bit s of
// 64-bit per-vertex masks:
//  - BFS: seen[v] holds the sources that reached v; F[L][v] the sources for
//    which v is at level L.  A level step expands every frontier vertex u
//    once for all its sources: per edge (u, v) new = F[L][u] & ~seen[v] is
//    claimed with one 64-bit atomicOr, so 64 BFS advance together.  Every
//    frontier entry (v, F[L][v]) stays in an append-only per-level log, from
//    which the distances of one source are materialised on demand (each
//    (v, s) bit is set at exactly one level).
//  - SSSP: dist is stored source-minor (dist[v * 64 + s]) so the 64 lanes of
//    a wave relax one edge for all sources with one coalesced 256-byte
//    access; F[i][v] holds the sources whose distance to v improved in
//    step i (label-correcting, as the single-source SSSP).
// Frontier bookkeeping follows the single-source traversal: counters in
// three rotating slots read on the device, hub vertices (more than
// kMsSmall buckets) listed one entry per kHubChunk buckets and spread over
// all waves, and the
// host reading counters only every few steps.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "profile.hpp"
#include "readback.hpp"
#include "slabhash.hpp"

namespace mk {

constexpr uint32_t kMsSmall = 2;

// BFS rotates three slots (its queue is the append-only log); SSSP rotates
// four, because a step clears the masks of the previous queue (slot i-1)
// and the counters of the one before (slot i-2).
constexpr uint32_t kMsSlots = 4;

constexpr uint32_t kMsStats = 16;

struct alignas(64) MsCounts {
  uint32_t cnt[kMsSlots];          // small entries per slot
  uint32_t steps;                  // non-empty steps
  uint32_t pad0;
  unsigned long long large[kMsSlots];  // (hub-list entries << 32) | buckets per slot
  uint32_t overflow;               // log capacity exceeded
  uint32_t pad;
  // per slot: the sources with an entry in that slot's queue (the OR of the
  // bits the step writing it set, and of admissions into it); a source
  // missing from the queue of the next step has converged
  unsigned long long active[kMsSlots];
  uint32_t scan[kMsSlots];  // SSSP: slots whose frontier is only its masks (no queue)
  // totals over kMsStats lines
  struct alignas(64) Stat {
    unsigned long long edges;  // adjacency entries read
    unsigned long long slabs;  // slabs read
    unsigned long long pairs;  // SSSP: (entry, active source) relaxations examined
    uint32_t width[kMsSlots];  // SSSP, per slot: the buckets a scan expanded
  } stat[kMsStats];
};

struct MsView {
  uint64_t *seen;      // BFS
  uint64_t *F[kMsSlots];  // per-step masks
  uint32_t *dist;      // SSSP, n * 64
  uint32_t *logv;      // BFS log / SSSP queues (kMsSlots * n)
  uint64_t *logm;      // BFS log masks
  uint32_t *seg;       // BFS: first log index of each level
  uint32_t log_cap;
  uint2 *ql[kMsSlots];  // hub lists
  MsCounts *c;
  uint32_t *off;       // BFS: level at which each source slot was admitted
  uint32_t n;
};

MK_DEV uint64_t wave_or64(uint64_t x) {
  for (int o = 32; o >= 1; o >>= 1) {
    const uint32_t lo = uint32_t(__shfl_xor(int(uint32_t(x)), o, 64));
    const uint32_t hi = uint32_t(__shfl_xor(int(uint32_t(x >> 32)), o, 64));
    x |= (uint64_t(hi) << 32) | lo;
  }
  return x;
}

MK_DEV uint64_t read_lane64(uint64_t x, uint32_t l) {
  return (uint64_t(read_lane(uint32_t(x >> 32), l)) << 32) | read_lane(uint32_t(x), l);
}

constexpr uint32_t kMsWaveQ = 512;  // LDS staging entries per wave

// Per-wave LDS staging of list appends: one global atomicAdd per flush.
struct MsQ {
  uint32_t *buf;
  uint32_t n;  // wave-uniform
};

MK_DEV void ms_flush(const MsView &S, MsQ &q, uint32_t *list, uint32_t base, uint32_t *cnt,
                     uint32_t cap) {
  if (q.n == 0) return;
  __builtin_amdgcn_wave_barrier();
  uint32_t pos = 0;
  if (lane_id() == 0) pos = atomicAdd(cnt, q.n);
  pos = read_lane(pos, 0);
  for (uint32_t i = lane_id(); i < q.n; i += 64) {
    if (base + pos + i < cap) list[base + pos + i] = q.buf[i];
    else atomicOr(&S.c->overflow, 1u);
  }
  __builtin_amdgcn_wave_barrier();
  q.n = 0;
}

// Append v (lanes with `push`) to the list (through the wave's staging) and
// hub vertices also to the hub list `ql` / `large`; `log_all` keeps hubs in
// the list too.  Entries past `cap` set the overflow flag instead of being
// written.  Wave-collective.
MK_DEV void ms_push(const GraphView &G, const MsView &S, MsQ &q, bool push, uint32_t v,
                    uint32_t *list, uint32_t base, uint32_t *cnt, uint2 *ql,
                    unsigned long long *large, uint32_t cap, bool log_all) {
  const uint64_t pm = ballot(push);
  if (pm == 0) return;
  uint32_t nb = 0;
  if (push) nb = G.bucket_off[v + 1] - G.bucket_off[v];
  const bool hub = push && nb > kMsSmall;
  const bool to_list = push && (log_all || !hub);
  const uint64_t lm = ballot(to_list);
  const uint32_t c = uint32_t(__popcll(lm));
  if (q.n + c > kMsWaveQ) ms_flush(S, q, list, base, cnt, cap);
  if (to_list) q.buf[q.n + lanes_below(lm)] = v;
  q.n += c;
  push_hubs(G, ql, large, hub, v, nb);
}

// A step's totals: one add a block, spread over lines (adds to one line are
// applied one after another, some 8 ns each: three a wave took 110 us of
// every step).  `acc` is wave-uniform.  Block-collective, once per kernel.
MK_DEV void add_totals(const MsView &S, uint32_t slot, uint32_t nslot, uint32_t edges,
                       uint32_t slabs, uint64_t pairs, uint32_t width, uint64_t acc) {
  __shared__ unsigned long long tot[3];
  __shared__ uint32_t totw;
  if (threadIdx.x < 3) tot[threadIdx.x] = 0ull;
  if (threadIdx.x == 3) totw = 0u;
  __syncthreads();
  if (lane_id() == 0 && slabs) {
    atomicAdd(&tot[0], (unsigned long long)edges);
    atomicAdd(&tot[1], (unsigned long long)slabs);
    atomicAdd(&tot[2], (unsigned long long)pairs);
    if (width) atomicAdd(&totw, width);
  }
  // (most waves find their bits set already)
  if (lane_id() == 0 && (acc & ~*(volatile unsigned long long *)&S.c->active[nslot]))
    atomicOr(&S.c->active[nslot], (unsigned long long)acc);
  __syncthreads();
  MsCounts::Stat &st = S.c->stat[blockIdx.x % kMsStats];
  if (threadIdx.x == 0 && tot[1]) {
    atomicAdd(&st.edges, tot[0]);
    atomicAdd(&st.slabs, tot[1]);
    if (tot[2]) atomicAdd(&st.pairs, tot[2]);
    if (totw) atomicAdd(&st.width[slot], totw);
  }
}

// ------------------------------------------------------------------ BFS
// BFS work on one slab of u (mask mu): each neighbour takes the source bits
// of mu it has not seen before this level; a vertex entering level L+1 is
// pushed once (first bits).  The seen update does not return: two waves
// that both take bit s of x in this level both put it into the same level's
// mask, so each (vertex, source) bit still lands in exactly one level.
MK_DEV void msbfs_slab(const GraphView &G, const MsView &S, MsQ &q, uint64_t key_mask_all,
                       uint32_t x, uint64_t mu, uint64_t *Fn, uint32_t nbase, uint32_t nslot,
                       uint32_t &edges, uint64_t &acc) {
  const uint32_t lane = lane_id();
  const bool live = ((key_mask_all >> lane) & 1ull) && x < kTomb;
  edges += uint32_t(__popcll(ballot(live)));
  bool push = false;
  if (live) {
    const uint64_t nw = mu & ~S.seen[x];
    if (nw) {
      atomicOr((unsigned long long *)(S.seen + x), (unsigned long long)nw);
      acc |= nw;
      push = atomicOr((unsigned long long *)(Fn + x), (unsigned long long)nw) == 0;
    }
  }
  ms_push(G, S, q, push, x, S.logv, nbase, &S.c->cnt[nslot], S.ql[nslot], &S.c->large[nslot],
          S.log_cap, true);
}

template <bool MAP>
MK_DEV void msbfs_chain(const GraphView &G, const MsView &S, MsQ &q, uint32_t x, uint64_t mu,
                        uint64_t *Fn, uint32_t nbase, uint32_t nslot, uint32_t &edges,
                        uint32_t &slabs, uint64_t &acc) {
  for (;;) {
    ++slabs;
    msbfs_slab(G, S, q, key_mask<MAP>(), x, mu, Fn, nbase, nslot, edges, acc);
    const uint32_t nx = read_lane(x, kNextLane);
    if (nx == kEmpty) break;
    x = slab_ptr(G.pool, nx)[lane_id()];
  }
}

// Level L: log segment [seg[L], seg[L] + cnt[L%3]) plus the hub list of
// slot L%3.  Appends to the log after it and to the hub list of slot
// (L+1)%3; clears slot (L+2)%3 and the masks of level L-1.
template <bool MAP>
__global__ void __launch_bounds__(kBlock) k_msbfs_level(GraphView G, MsView S, uint32_t L) {
  const uint32_t lane = lane_id();
  const uint32_t gw = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t W = (gridDim.x * blockDim.x) >> 6;
  const uint32_t slot = L % 3, nslot = (L + 1) % 3, pslot = (L + 2) % 3;
  const uint32_t start = S.seg[L];
  const uint32_t count = S.c->cnt[slot];
  const uint32_t nbase = start + count;
  const unsigned long long lg = S.c->large[slot];
  const uint32_t n_large = uint32_t(lg >> 32);  // hub-list entries
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    S.seg[L + 1] = nbase;
    S.c->cnt[pslot] = 0;
    S.c->large[pslot] = 0ull;
    S.c->active[pslot] = 0ull;
    if (count) atomicAdd(&S.c->steps, 1u);
  }
  uint64_t *Fc = S.F[slot], *Fn = S.F[nslot], *Fp = S.F[pslot];
  // masks of level L-1 are no longer read: clear them for level L+2 (also
  // when level L is empty: a source admitted later makes level L+1 run, and
  // level L+2's masks must then start clear)
  if (L > 0) {
    const uint32_t ps = S.seg[L - 1];
    for (uint32_t i = ps + gw * 64 + lane; i < min(start, S.log_cap); i += W * 64)
      Fp[S.logv[i]] = 0ull;
  }
  if (count == 0) return;
  // after a log overflow (the run is repeated) only stored entries are read
  const uint32_t end = min(nbase, S.log_cap);
  __shared__ uint32_t lqbuf[kBlock / 64][kMsWaveQ];
  MsQ q{lqbuf[threadIdx.x >> 6], 0u};
  uint32_t edges = 0, slabs = 0;
  uint64_t acc = 0;  // source bits this lane set in the next level's masks
  // hubs: their list entries
  const uint2 *ql = S.ql[slot];
  // lane l takes bucket l % kHubChunk of hub-list entry l / kHubChunk
  const uint32_t eper = min(per_wave(n_large, W), 64u / kHubChunk);
  for (uint32_t e0 = gw * eper; e0 < n_large; e0 += W * eper) {
    const uint32_t el = lane / kHubChunk, ei = e0 + el;
    bool act = el < eper && ei < n_large;
    uint32_t b = 0;
    uint64_t mu = 0;
    if (act) {
      const uint2 ent = ql[ei];
      b = ent.y + lane % kHubChunk;
      act = b < G.bucket_off[ent.x + 1];
      if (act) mu = Fc[ent.x];
    }
    uint64_t m = ballot(act);
    while (m) {
      uint32_t js[4];
      uint32_t c = 0;
#pragma unroll
      for (uint32_t qq = 0; qq < 4; ++qq) {
        js[qq] = m ? ffs64(m) : 0u;
        if (m) {
          m &= m - 1;
          c = qq + 1;
        }
      }
      uint32_t x[4];
#pragma unroll
      for (uint32_t qq = 0; qq < 4; ++qq)
        x[qq] = qq < c ? G.heads[size_t(read_lane(b, js[qq])) * kSlabWords + lane] : kEmpty;
#pragma unroll
      for (uint32_t qq = 0; qq < 4; ++qq)
        if (qq < c)
          msbfs_chain<MAP>(G, S, q, x[qq], read_lane64(mu, js[qq]), Fn, nbase, nslot, edges, slabs,
                           acc);
    }
  }
  // log entries: record the mask; expand non-hub vertices
  const uint32_t per = per_wave(end - start, W);
  for (uint32_t i0 = start + gw * per; i0 < end; i0 += W * per) {
    const uint32_t i = i0 + lane;
    bool act = lane < per && i < end;
    uint32_t u = 0, b0 = 0, nb = 0;
    uint64_t mu = 0;
    if (act) {
      u = S.logv[i];
      mu = Fc[u];
      S.logm[i] = mu;
      b0 = G.bucket_off[u];
      nb = G.bucket_off[u + 1] - b0;
      if (nb > kMsSmall) act = false;
    }
    for (uint32_t k = 0; ballot(act && nb > k); ++k) {
      uint64_t m = ballot(act && nb > k);
      while (m) {
        uint32_t js[4];
        uint32_t c = 0;
#pragma unroll
        for (uint32_t qq = 0; qq < 4; ++qq) {
          js[qq] = m ? ffs64(m) : 0u;
          if (m) {
            m &= m - 1;
            c = qq + 1;
          }
        }
        uint32_t x[4];
#pragma unroll
        for (uint32_t qq = 0; qq < 4; ++qq)
          x[qq] = qq < c ? G.heads[size_t(read_lane(b0, js[qq]) + k) * kSlabWords + lane] : kEmpty;
#pragma unroll
        for (uint32_t qq = 0; qq < 4; ++qq)
          if (qq < c)
            msbfs_chain<MAP>(G, S, q, x[qq], read_lane64(mu, js[qq]), Fn, nbase, nslot, edges,
                             slabs, acc);
      }
    }
  }
  ms_flush(S, q, S.logv, nbase, &S.c->cnt[nslot], S.log_cap);
  add_totals(S, slot, nslot, edges, slabs, 0, 0, wave_or64(acc));
}

// The first frontier, a lane per source (one wave; sources may repeat: the
// same vertex in two slots).  64 sources, against one thread taking them in
// turn: 41 -> 3 us.
__global__ void __launch_bounds__(64) k_ms_init(MsView S, const uint32_t *sources, uint32_t k,
                                                uint32_t sssp) {
  const uint32_t s = threadIdx.x;
  uint32_t v = 0;
  bool fresh = false;
  if (s < k) {
    const unsigned long long bit = 1ull << s;
    v = sources[s];
    fresh = atomicOr((unsigned long long *)(S.F[0] + v), bit) == 0;
    if (sssp) S.dist[size_t(v) * 64 + s] = 0;
    else atomicOr((unsigned long long *)(S.seen + v), bit);
  }
  const uint64_t m = ballot(fresh);
  if (fresh) S.logv[lanes_below(m)] = v;
  if (s == 0) {
    if (!sssp) S.seg[0] = 0;
    S.c->cnt[0] = uint32_t(__popcll(m));
  }
}

// Hub vertices among the sources go to the hub list of slot 0 (one wave).
__global__ void k_ms_source_hubs(GraphView G, MsView S) {
  const uint32_t i = threadIdx.x;
  uint32_t v = 0, nb = 0;
  if (i < S.c->cnt[0]) {
    v = S.logv[i];
    nb = G.bucket_off[v + 1] - G.bucket_off[v];
  }
  push_hubs(G, S.ql[0], &S.c->large[0], nb > kMsSmall, v, nb);
}

// Distances of slot s from the log: the level whose mask holds bit s.
__global__ void k_msbfs_read(MsView S, uint32_t s, uint32_t total, uint32_t levels,
                             uint32_t *out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  if (!((S.logm[i] >> s) & 1ull)) return;
  uint32_t lo = 0, hi = levels;  // last level with seg <= i
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (S.seg[mid] <= i) lo = mid;
    else hi = mid;
  }
  out[S.logv[i]] = lo - S.off[s];
}

// ------------------------------------------------------------------ SSSP
// A frontier vertex with at most this many active sources relaxes its slabs
// key-parallel (lanes = neighbours, one pass per source) instead of
// row-parallel (lanes = sources, neighbours a few at a time).
constexpr uint32_t kMsSparse = 4;
// Neighbours' distance rows a scan step keeps in flight per wave: 24 waves a
// CU of them already draw all that memory gives for random 256-byte rows
// (RMAT-20, 64 sources, a run's steps: 5.2 ms with 4 rows; 5.9 with 2, 5.4
// with 3, 5.8 with 8, 7.6 with 16).
constexpr uint32_t kMsScanRows = 4;

// Relax one slab of u for all sources in mu: per live key (neighbour v,
// weight w), lanes are sources; U neighbours' distance rows are loaded at a
// time.  Neither the minimum nor (with `push` off) the mask update waits for
// an old value: a candidate below the distance read marks its source bit
// whether or not its own minimum lands last.  That sets no bit too many: a
// distance read is never above the one the step began with, so some
// candidate of this step improves it.  With `push`, a neighbour whose mask
// was empty before is appended to the next queue.
template <bool MAP, uint32_t U>
MK_DEV void mssp_slab(const GraphView &G, const MsView &S, MsQ &q, uint32_t x, uint32_t du_lane,
                      uint64_t mu, uint64_t *Fn, uint32_t *qn, uint32_t nslot, bool push,
                      uint32_t &edges, uint64_t &pairs, uint64_t &acc) {
  const uint32_t lane = lane_id();
  const uint64_t km = key_mask<MAP>();
  uint64_t live = ballot(x < kTomb) & km;
  edges += uint32_t(__popcll(live));
  pairs += uint64_t(__popcll(live)) * uint64_t(__popcll(mu));
  if (uint32_t(__popcll(mu)) <= kMsSparse) {
    // key-parallel: lane j relaxes key j of this slab for each active source
    const bool lv = (live >> lane) & 1ull;
    const uint32_t wv = MAP ? __shfl_down(x, 1, 64) : 1u;
    for (uint64_t m = mu; m; m &= m - 1) {
      const uint32_t src = ffs64(m);
      const uint32_t du = read_lane(du_lane, src);
      if (du == kInf) continue;
      bool fresh = false, imp = false;
      if (lv) {
        const uint32_t cand = du + wv;
        uint32_t *dp = S.dist + size_t(x) * 64 + src;
        imp = cand >= du && cand < *dp;
        if (imp) {
          (void)atomicMin(dp, cand);
          unsigned long long *fp = (unsigned long long *)(Fn + x);
          if (push) fresh = atomicOr(fp, 1ull << src) == 0;
          else (void)atomicOr(fp, 1ull << src);
        }
      }
      if (ballot(imp)) acc |= 1ull << src;
      if (push)
        ms_push(G, S, q, fresh, x, qn, 0, &S.c->cnt[nslot], S.ql[nslot], &S.c->large[nslot], S.n,
                false);
    }
    return;
  }
  // only the lanes of sources active at u read their distance word, so a
  // sparse mask touches one line of the 256-byte row, not both
  const bool reads = ((mu >> lane) & 1ull) && du_lane != kInf;
  uint64_t mine = 0;  // the sources improved at this lane's key
  while (live) {
    uint32_t ks[U], v[U], cur[U];
    uint32_t c = 0;
#pragma unroll
    for (uint32_t qq = 0; qq < U; ++qq) {
      ks[qq] = v[qq] = 0u;
      if (live) {
        ks[qq] = ffs64(live);
        live &= live - 1;
        v[qq] = read_lane(x, ks[qq]);
        c = qq + 1;
      }
    }
#pragma unroll
    for (uint32_t qq = 0; qq < U; ++qq) cur[qq] = 0u;
    if (reads) {
#pragma unroll
      for (uint32_t qq = 0; qq < U; ++qq)
        if (qq < c) cur[qq] = S.dist[size_t(v[qq]) * 64 + lane];
    }
#pragma unroll
    for (uint32_t qq = 0; qq < U; ++qq) {
      if (qq < c) {
        // du + w < cur without overflow
        const uint32_t w = MAP ? read_lane(x, ks[qq] + 1) : 1u;
        const bool imp = w < __builtin_elementwise_sub_sat(cur[qq], du_lane);
        const uint64_t im = ballot(imp);
        if (im) {
          if (imp) (void)atomicMin(S.dist + size_t(v[qq]) * 64 + lane, du_lane + w);
          acc |= im;
          if (lane == ks[qq]) mine = im;
        }
      }
    }
  }
  // one mask update for the slab: lane k its key's
  if (ballot(mine != 0) == 0) return;
  unsigned long long *fp = (unsigned long long *)(Fn + x);
  if (push) {
    bool fresh = false;
    if (mine) fresh = atomicOr(fp, (unsigned long long)mine) == 0;
    ms_push(G, S, q, fresh, x, qn, 0, &S.c->cnt[nslot], S.ql[nslot], &S.c->large[nslot], S.n,
            false);
  } else if (mine) {
    (void)atomicOr(fp, (unsigned long long)mine);
  }
}

template <bool MAP, uint32_t U>
MK_DEV void mssp_chain(const GraphView &G, const MsView &S, MsQ &q, uint32_t x, uint32_t du,
                       uint64_t mu, uint64_t *Fn, uint32_t *qn, uint32_t nslot, bool push,
                       uint32_t &edges, uint32_t &slabs, uint64_t &pairs, uint64_t &acc) {
  for (;;) {
    ++slabs;
    mssp_slab<MAP, U>(G, S, q, x, du, mu, Fn, qn, nslot, push, edges, pairs, acc);
    const uint32_t nx = read_lane(x, kNextLane);
    if (nx == kEmpty) break;
    x = slab_ptr(G.pool, nx)[lane_id()];
  }
}

// A step whose frontier has at least 1/kMsDense of the graph's buckets goes
// over all buckets, looking up each one's mask, and leaves its next frontier
// as masks alone: no queue, so no update waits for an old value (the queue
// form waits for the minimum, the mask and the list position in turn).
// RMAT-20, 64 sources: a step over all 16M edges 2.6 -> 1.0 ms, a run's steps
// 13.4 -> 5.2 ms; bounded by the rows read past the L2 (3.2 GB a step).  The
// least such frontier reads about what the scan's owner and mask words do.
constexpr uint32_t kMsDense = 16;
// Buckets a wave takes at a time (fewer even out the waves' work, and cost
// owner and mask reads; 4, 6 and 8 were within 1% at RMAT-20, 4 the best by
// 4-10% at RMAT-15 to 19).
constexpr uint32_t kMsTake = 4;

// The scan form of a step: every bucket whose vertex has sources in Fc.
template <bool MAP>
MK_DEV void mssp_scan(const GraphView &G, const MsView &S, MsQ &q, uint32_t gw, uint32_t W,
                      const uint64_t *Fc, uint64_t *Fn, uint32_t *qn, uint32_t nslot, bool push,
                      uint32_t &width, uint32_t &edges, uint32_t &slabs, uint64_t &pairs,
                      uint64_t &acc) {
  const uint32_t lane = lane_id();
  const uint32_t T = G.total_buckets;
  const uint32_t per = min(per_wave(T, W), kMsTake);
  for (uint64_t k0 = uint64_t(gw) * per; k0 < T; k0 += uint64_t(W) * per) {
    const uint64_t k = k0 + lane;
    uint32_t u = 0;
    uint64_t mu = 0;
    if (lane < per && k < T) {
      u = G.bucket_owner[k];
      mu = Fc[u];
    }
    uint64_t m = ballot(mu != 0);
    width += uint32_t(__popcll(m));
    while (m) {
      uint32_t js[4], x[4], du[4];
      uint32_t c = 0;
#pragma unroll
      for (uint32_t qq = 0; qq < 4; ++qq) {
        js[qq] = 0u;
        x[qq] = kEmpty;
        du[qq] = kInf;
        if (m) {
          js[qq] = ffs64(m);
          m &= m - 1;
          c = qq + 1;
          x[qq] = G.heads[size_t(k0 + js[qq]) * kSlabWords + lane];
          du[qq] = S.dist[size_t(read_lane(u, js[qq])) * 64 + lane];
        }
      }
#pragma unroll 1
      for (uint32_t qq = 0; qq < c; ++qq) {
        const uint32_t xq = qq == 0 ? x[0] : qq == 1 ? x[1] : qq == 2 ? x[2] : x[3];
        const uint32_t dq = qq == 0 ? du[0] : qq == 1 ? du[1] : qq == 2 ? du[2] : du[3];
        const uint32_t jq = qq == 0 ? js[0] : qq == 1 ? js[1] : qq == 2 ? js[2] : js[3];
        mssp_chain<MAP, kMsScanRows>(G, S, q, xq, dq, read_lane64(mu, jq), Fn, qn, nslot, push,
                                     edges, slabs, pairs, acc);
      }
    }
  }
}

// The queue form of a step: the hub list's buckets, then the small vertices.
template <bool MAP, uint32_t U>
MK_DEV void mssp_queue(const GraphView &G, const MsView &S, MsQ &q, uint32_t gw, uint32_t W,
                       uint32_t slot, uint32_t nslot, uint32_t count, uint32_t n_large,
                       uint32_t &edges, uint32_t &slabs, uint64_t &pairs, uint64_t &acc) {
  const uint32_t lane = lane_id();
  const uint32_t *qc = S.logv + size_t(slot) * S.n;
  uint32_t *qn = S.logv + size_t(nslot) * S.n;
  const uint64_t *Fc = S.F[slot];
  uint64_t *Fn = S.F[nslot];
  const uint2 *ql = S.ql[slot];
  // lane l takes bucket l % kHubChunk of hub-list entry l / kHubChunk
  const uint32_t eper = min(per_wave(n_large, W), 64u / kHubChunk);
  for (uint32_t e0 = gw * eper; e0 < n_large; e0 += W * eper) {
    const uint32_t el = lane / kHubChunk, ei = e0 + el;
    bool act = el < eper && ei < n_large;
    uint32_t b = 0, u = 0;
    uint64_t mu = 0;
    if (act) {
      const uint2 ent = ql[ei];
      u = ent.x;
      b = ent.y + lane % kHubChunk;
      act = b < G.bucket_off[u + 1];
      if (act) mu = Fc[u];
    }
    uint64_t m = ballot(act);
    while (m) {
      uint32_t js[4];
      uint32_t c = 0;
#pragma unroll
      for (uint32_t qq = 0; qq < 4; ++qq) {
        js[qq] = m ? ffs64(m) : 0u;
        if (m) {
          m &= m - 1;
          c = qq + 1;
        }
      }
      uint32_t x[4];
#pragma unroll
      for (uint32_t qq = 0; qq < 4; ++qq)
        x[qq] = qq < c ? G.heads[size_t(read_lane(b, js[qq])) * kSlabWords + lane] : kEmpty;
      // one copy of the expansion for the four heads (their loads above are
      // already in flight): fewer registers than four inlined copies
#pragma unroll 1
      for (uint32_t qq = 0; qq < c; ++qq) {
        const uint32_t xq = qq == 0 ? x[0] : qq == 1 ? x[1] : qq == 2 ? x[2] : x[3];
        const uint32_t jq = qq == 0 ? js[0] : qq == 1 ? js[1] : qq == 2 ? js[2] : js[3];
        const uint32_t du = S.dist[size_t(read_lane(u, jq)) * 64 + lane];
        mssp_chain<MAP, U>(G, S, q, xq, du, read_lane64(mu, jq), Fn, qn, nslot, true, edges, slabs,
                           pairs, acc);
      }
    }
  }
  const uint32_t per = per_wave(count, W);
  for (uint32_t k0 = gw * per; k0 < count; k0 += W * per) {
    const uint32_t k = k0 + lane;
    bool act = lane < per && k < count;
    uint32_t u = 0, b0 = 0, nb = 0;
    uint64_t mu = 0;
    if (act) {
      u = qc[k];
      mu = Fc[u];
      b0 = G.bucket_off[u];
      nb = G.bucket_off[u + 1] - b0;
      if (nb > kMsSmall) act = false;  // hubs are expanded from the hub list
    }
    for (uint32_t kk = 0; ballot(act && nb > kk); ++kk) {
      uint64_t m = ballot(act && nb > kk);
      while (m) {
        const uint32_t j = ffs64(m);
        m &= m - 1;
        const uint32_t x = G.heads[size_t(read_lane(b0, j) + kk) * kSlabWords + lane];
        const uint32_t du = S.dist[size_t(read_lane(u, j)) * 64 + lane];
        mssp_chain<MAP, U>(G, S, q, x, du, read_lane64(mu, j), Fn, qn, nslot, true, edges, slabs,
                           pairs, acc);
      }
    }
  }
}

// SSSP step i: the frontier of slot i%4 (masks F[i%4], and, unless scan[i%4],
// its queue); leaves that of slot (i+1)%4; clears the masks of slot (i+3)%4
// (step i-1's) and the counters of slot (i+2)%4 (queue i-2, whose masks step
// i-1 cleared).
template <bool MAP, uint32_t U>
__global__ void __launch_bounds__(kBlock) k_mssp_step(GraphView G, MsView S, uint32_t i) {
  const uint32_t lane = lane_id();
  const uint32_t gw = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t W = (gridDim.x * blockDim.x) >> 6;
  const uint32_t slot = i % kMsSlots, nslot = (i + 1) % kMsSlots;
  const uint32_t zslot = (i + 2) % kMsSlots, pslot = (i + 3) % kMsSlots;
  const uint32_t count = S.c->cnt[slot];
  const unsigned long long lg = S.c->large[slot];
  const uint32_t n_large = uint32_t(lg >> 32);  // hub-list entries
  uint32_t *qn = S.logv + size_t(nslot) * S.n;
  const uint32_t *qp = S.logv + size_t(pslot) * S.n;
  uint64_t *Fc = S.F[slot], *Fn = S.F[nslot], *Fp = S.F[pslot];
  const bool masks = S.c->scan[slot] != 0;  // no queue was kept
  const bool none = masks ? S.c->active[slot] == 0 : count + n_large == 0;
  // buckets of this frontier (of one without a queue: as wide as the last)
  uint64_t wide = uint64_t(count) + uint32_t(lg);
  if (masks) {
    const uint32_t wl = lane < kMsStats ? S.c->stat[lane].width[pslot] : 0u;
    wide = wave_sum_u32(wl);
  }
  const bool dense = !none && wide * kMsDense >= G.total_buckets;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    S.c->cnt[zslot] = 0;
    S.c->large[zslot] = 0ull;
    S.c->active[zslot] = 0ull;
    S.c->scan[nslot] = dense ? 1u : 0u;
  }
  if (blockIdx.x == 0 && threadIdx.x < kMsStats) S.c->stat[threadIdx.x].width[zslot] = 0u;
  // step i-1 is done: clear its masks before its slot is reused
  if (i > 0 && S.c->scan[pslot]) {
    for (uint32_t k = gw * 64 + lane; k < S.n; k += W * 64) Fp[k] = 0ull;
  } else if (i > 0) {
    const uint32_t pcount = S.c->cnt[pslot];
    const uint32_t plarge = uint32_t(S.c->large[pslot] >> 32);
    for (uint32_t k = gw * 64 + lane; k < pcount; k += W * 64) Fp[qp[k]] = 0ull;
    for (uint32_t k = gw * 64 + lane; k < plarge; k += W * 64) Fp[S.ql[pslot][k].x] = 0ull;
  }
  if (none) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) atomicAdd(&S.c->steps, 1u);
  __shared__ uint32_t lqbuf[kBlock / 64][kMsWaveQ];
  MsQ q{lqbuf[threadIdx.x >> 6], 0u};
  uint32_t edges = 0, slabs = 0;
  uint64_t pairs = 0, acc = 0;  // acc: source bits improved into the next queue
  uint32_t width = 0;
  if (masks || dense) {
    mssp_scan<MAP>(G, S, q, gw, W, Fc, Fn, qn, nslot, !dense, width, edges, slabs, pairs, acc);
  } else {
    mssp_queue<MAP, U>(G, S, q, gw, W, slot, nslot, count, n_large, edges, slabs, pairs, acc);
  }
  ms_flush(S, q, qn, 0, &S.c->cnt[nslot], S.n);
  add_totals(S, slot, nslot, edges, slabs, pairs, width, acc);
}

// Sources admitted into free slots of a running traversal (continuous
// batching), before step `step`: the sources join that step's frontier
// (queue slot `qs`: step % kMsSlots for SSSP, step % 3 for BFS) and their
// bits mark the slot active.  SSSP: distance 0 in the source's lane.  BFS:
// the source's bit in seen; its level 0 is `step`, recorded in off[slot].
// Passed by value: no copy to stage.
struct MsAdmit {
  uint32_t v[64];
  uint32_t slot[64];
  uint32_t k;
};

// One wave: lane 0 appends in order (a vertex named twice, or already in
// the frontier, is queued once), then the new hub vertices go to the hub
// list together.
__global__ void __launch_bounds__(64) k_ms_admit(GraphView G, MsView S, MsAdmit a, uint32_t step,
                                                 uint32_t sssp) {
  __shared__ uint32_t fresh[64];
  const uint32_t t = threadIdx.x;
  const uint32_t qs = sssp ? step % kMsSlots : step % 3;
  if (t == 0) {
    uint32_t cnt = S.c->cnt[qs];
    const uint32_t base = sssp ? qs * S.n : S.seg[step];
    uint64_t act = 0;
    for (uint32_t i = 0; i < a.k; ++i) {
      const uint32_t v = a.v[i], s = a.slot[i];
      const uint64_t bit = 1ull << s;
      fresh[i] = 0u;
      if (S.F[qs][v] == 0) {
        if (sssp || base + cnt < S.log_cap) S.logv[base + cnt] = v;
        else S.c->overflow = 1u;
        ++cnt;
        fresh[i] = 1u;
      }
      S.F[qs][v] |= bit;
      if (sssp) {
        S.dist[size_t(v) * 64 + s] = 0;
      } else {
        S.seen[v] |= bit;
        S.off[s] = step;
      }
      act |= bit;
    }
    S.c->cnt[qs] = cnt;
    S.c->active[qs] |= act;
  }
  __syncthreads();
  uint32_t v = 0, nb = 0;
  bool hub = false;
  if (t < a.k && fresh[t]) {
    v = a.v[t];
    nb = G.bucket_off[v + 1] - G.bucket_off[v];
    hub = nb > kMsSmall;
  }
  push_hubs(G, S.ql[qs], &S.c->large[qs], hub, v, nb);
}

// ------------------------------------------------------------------ host
struct MultiSource {
  mk_graph *g = nullptr;
  bool sssp = false;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  uint64_t *seen = nullptr;
  uint64_t *F[kMsSlots] = {nullptr, nullptr, nullptr, nullptr};
  uint32_t *dist = nullptr;
  uint32_t *logv = nullptr;
  uint64_t *logm = nullptr;
  uint32_t *seg = nullptr;
  uint32_t log_cap = 0;
  uint2 *ql[kMsSlots] = {nullptr, nullptr, nullptr, nullptr};
  MsCounts *c = nullptr;
  uint32_t *src_dev = nullptr;
  uint32_t *off = nullptr;  // BFS: admission level per slot
  HostBuf host;
  DevBuf read_buf;          // BFS: one slot's distances, scattered from the log
  // continuous batching (open / admit / launch / poll): the session's next
  // step, the slots admitted since open, and whether a session is open
  bool session = false;
  bool grow_log = false;  // a session's log filled up: the next one gets a larger log
  uint32_t step = 0;
  uint64_t admitted = 0;
  uint32_t k = 0;
  uint32_t last_steps = 0;
  uint64_t last_edges = 0;
  uint32_t log_total = 0;
  int max_waves = 0;
  int unroll = 4;

  MsView view() const {
    MsView v;
    v.seen = seen;
    for (uint32_t i = 0; i < kMsSlots; ++i) {
      v.F[i] = F[i];
      v.ql[i] = ql[i];
    }
    v.dist = dist;
    v.logv = logv;
    v.logm = logm;
    v.seg = seg;
    v.log_cap = log_cap;
    v.c = c;
    v.off = off;
    v.n = g->n;
    return v;
  }

  // BFS level log of `entries` (vertex, mask) entries; no run or session
  // needs more than 64 per vertex (each source bit of a vertex is set at one
  // level) plus the admissions
  int alloc_log(uint64_t entries) {
    (void)hipFree(logv);
    (void)hipFree(logm);
    logv = nullptr;
    logm = nullptr;
    entries = std::min<uint64_t>(entries, 64 * uint64_t(g->n) + 64);
    entries = std::min<uint64_t>(entries, 0xFFFFFFF0ull);
    MK_HIP(hipMalloc(&logv, entries * 4));
    MK_HIP(hipMalloc(&logm, entries * 8));
    log_cap = uint32_t(entries);
    return MK_OK;
  }

  int init(mk_graph *graph, bool is_sssp) {
    g = graph;
    sssp = is_sssp;
    const size_t n = g->n;
    MK_HIP(hipSetDevice(g->device));
    MK_HIP(hipStreamCreate(&stream));
    loop_stream_add(g->device, stream, 1);
    MK_HIP(hipEventCreate(&ev0));
    MK_HIP(hipEventCreate(&ev1));
    for (uint32_t i = 0; i < kMsSlots; ++i) {
      MK_HIP(hipMalloc(&F[i], n * 8));
      // one entry per kHubChunk buckets of each listed hub
      MK_HIP(hipMalloc(&ql[i], (n + size_t(g->total_buckets) / kHubChunk + 64) * 8));
      fill_u64(F[i], 0ull, n, stream);
    }
    MK_HIP(hipMalloc(&c, sizeof(MsCounts)));
    MK_HIP(hipMalloc(&src_dev, 64 * 4));
    MK_HIP(hipMalloc(&off, 64 * 4));
    if (sssp) {
      MK_HIP(hipMalloc(&dist, n * 64 * 4));
      MK_HIP(hipMalloc(&logv, kMsSlots * n * 4));  // one queue per slot
      log_cap = uint32_t(std::min<uint64_t>(kMsSlots * n, 0xFFFFFFF0ull));
    } else {
      MK_HIP(hipMalloc(&seen, n * 8));
      MK_HIP(hipMalloc(&seg, (n + 2) * 4));
      if (int r = alloc_log(8 * uint64_t(n) + 64)) return r;
    }
    if (int r = host.ensure(sizeof(MsCounts))) return r;
    MK_HIP(hipStreamSynchronize(stream));
    unroll = int(tune_get("ms_unroll", 8));
    if (int r = size_grid()) return r;
    return MK_OK;
  }

  void destroy() {
    (void)hipSetDevice(g->device);
    if (stream) (void)hipStreamSynchronize(stream);
    (void)hipFree(seen);
    for (uint32_t i = 0; i < kMsSlots; ++i) {
      (void)hipFree(F[i]);
      (void)hipFree(ql[i]);
    }
    (void)hipFree(dist);
    (void)hipFree(logv);
    (void)hipFree(logm);
    (void)hipFree(seg);
    (void)hipFree(c);
    (void)hipFree(src_dev);
    (void)hipFree(off);
    read_buf.release();
    host.release();
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) {
      loop_stream_add(g->device, stream, -1);
      (void)hipStreamDestroy(stream);
    }
  }

  // (the totals, summed, in h.stat[0])
  int read_counts(MsCounts &h) {
    MK_HIP(hipMemcpyAsync(host.ptr, c, sizeof(MsCounts), hipMemcpyDeviceToHost, stream));
    MK_HIP(hipStreamSynchronize(stream));
    h = *host.as<MsCounts>();
    for (uint32_t i = 1; i < kMsStats; ++i) {
      h.stat[0].edges += h.stat[i].edges;
      h.stat[0].slabs += h.stat[i].slabs;
      h.stat[0].pairs += h.stat[i].pairs;
    }
    return MK_OK;
  }

  // The step kernel this handle launches.
  const void *step_kernel() const {
    if (!sssp)
      return g->weighted ? reinterpret_cast<const void *>(&k_msbfs_level<true>)
                         : reinterpret_cast<const void *>(&k_msbfs_level<false>);
    return unroll == 8 ? reinterpret_cast<const void *>(&k_mssp_step<true, 8>)
                       : reinterpret_cast<const void *>(&k_mssp_step<true, 4>);
  }

  // The steps are latency-bound: `ms_waves_per_cu` waves per CU (more than
  // the frontier loops use keep more rows in flight), capped at what a CU
  // holds of the step kernel.
  int size_grid() {
    MK_HIP(resident_waves(g->device, step_kernel(), int(tune_get("ms_waves_per_cu", 24)),
                          &max_waves));
    return MK_OK;
  }

  void reset_state() {
    const size_t n = g->n;
    for (uint32_t i = 0; i < kMsSlots; ++i) fill_u64(F[i], 0ull, n, stream);
    fill_u32(reinterpret_cast<uint32_t *>(c), 0u, sizeof(MsCounts) / 4, stream);
    fill_u32(off, 0u, 64, stream);
    if (sssp) fill_u32(dist, kInf, n * 64, stream);
    else fill_u64(seen, 0ull, n, stream);
  }

  void launch_step(const GraphView &G, const MsView &S, uint32_t s, unsigned grid) {
    // multi-source SSSP needs a weighted graph (mk_msq_create): map slabs
    if (sssp) {
      if (unroll == 8) k_mssp_step<true, 8><<<grid, kBlock, 0, stream>>>(G, S, s);
      else k_mssp_step<true, 4><<<grid, kBlock, 0, stream>>>(G, S, s);
    } else {
      if (g->weighted) k_msbfs_level<true><<<grid, kBlock, 0, stream>>>(G, S, s);
      else k_msbfs_level<false><<<grid, kBlock, 0, stream>>>(G, S, s);
    }
  }

  // ---- continuous batching
  int open() {
    MK_HIP(hipSetDevice(g->device));
    if (grow_log) {
      MK_HIP(hipStreamSynchronize(stream));
      if (int r = alloc_log(uint64_t(log_cap) * 4)) return r;
      grow_log = false;
    }
    reset_state();
    if (!sssp) fill_u32(seg, 0u, 1, stream);  // level 0 starts the log
    MK_HIP(hipGetLastError());
    session = true;
    step = 0;
    admitted = 0;
    k = 0;
    last_steps = 0;
    last_edges = 0;
    return MK_OK;
  }

  int admit(const uint32_t *sources, const uint32_t *slots, uint32_t n) {
    if (!session) return fail(MK_ERR_STATE, "mk_msq_admit: no open session (mk_msq_open)");
    MsAdmit a;
    a.k = n;
    uint64_t bits = 0;
    for (uint32_t i = 0; i < n; ++i) {
      if (slots[i] >= 64) return fail(MK_ERR_BAD_ARG, "mk_msq_admit: slot >= 64");
      if (sources[i] >= g->n) return fail(MK_ERR_RANGE, "mk_msq_admit: source >= n");
      const uint64_t bit = 1ull << slots[i];
      if ((admitted | bits) & bit)
        return fail(MK_ERR_STATE, "mk_msq_admit: slot already used in this session");
      bits |= bit;
      a.v[i] = sources[i];
      a.slot[i] = slots[i];
    }
    if (n == 0) return MK_OK;
    if (!sssp && step + 1 >= g->n + 2) return fail(MK_ERR_STATE, "mk_msq_admit: session too long");
    MK_HIP(hipSetDevice(g->device));
    k_ms_admit<<<1, 64, 0, stream>>>(g->view(), view(), a, step, sssp ? 1u : 0u);
    MK_HIP(hipGetLastError());
    admitted |= bits;
    return MK_OK;
  }

  // Queue `steps` more steps of the session (they are no-ops once its
  // frontier is empty); poll() waits for them.
  int launch(uint32_t steps) {
    if (!session) return fail(MK_ERR_STATE, "mk_msq_launch: no open session (mk_msq_open)");
    MK_HIP(hipSetDevice(g->device));
    const GraphView G = g->view();
    const MsView S = view();
    const unsigned grid = blocks_for_waves(uint64_t(max_waves));
    for (uint32_t t = 0; t < steps; ++t, ++step) {
      ProfScope prof(stream, sssp ? "k_mssp_step" : "k_msbfs_level", 0.0);
      if (!sssp && step + 1 >= g->n + 2)
        return fail(MK_ERR_STATE, "multi-source BFS: session too long");
      launch_step(G, S, step, grid);
    }
    MK_HIP(hipGetLastError());
    return MK_OK;
  }

  // Wait for the queued steps; `active` = admitted slots with work left
  // (an admitted slot not in it has its final distances).
  int poll(uint64_t *active, uint32_t *steps_done) {
    if (!session) return fail(MK_ERR_STATE, "mk_msq_poll: no open session (mk_msq_open)");
    MsCounts h{};
    if (int r = read_counts(h)) return r;
    if (!sssp && h.overflow) {
      grow_log = true;
      return fail(MK_ERR_STATE, "multi-source BFS: the level log is full; the slots still "
                                "active are incomplete (open a new session for them: it gets a "
                                "log four times larger)");
    }
    last_steps = h.steps;
    last_edges = h.stat[0].edges;
    *active = h.active[step % (sssp ? kMsSlots : 3)] & admitted;
    if (steps_done) *steps_done = step;
    return MK_OK;
  }

  int run(const uint32_t *sources, uint32_t nsrc, float *ms) {
    MK_HIP(hipSetDevice(g->device));
    session = false;
    for (int attempt = 0; attempt < 4; ++attempt) {
      MK_HIP(hipEventRecord(ev0, stream));
      reset_state();
      MK_HIP(hipMemcpyAsync(src_dev, sources, nsrc * 4, hipMemcpyHostToDevice, stream));
      const GraphView G = g->view();
      const MsView S = view();
      k_ms_init<<<1, 64, 0, stream>>>(S, src_dev, nsrc, sssp ? 1u : 0u);
      k_ms_source_hubs<<<1, 64, 0, stream>>>(G, S);
      MK_HIP(hipGetLastError());
      const unsigned grid = blocks_for_waves(uint64_t(max_waves));
      uint32_t step = 0, group = 2;
      const uint64_t limit = uint64_t(g->n) * (sssp ? 1 : 64) + 8;
      MsCounts h{};
      for (;;) {
        for (uint32_t q = 0; q < group; ++q, ++step) {
          ProfScope prof(stream, sssp ? "k_mssp_step" : "k_msbfs_level", 0.0);
          if (!sssp && step + 1 >= g->n + 2) break;  // seg has n + 2 entries
          launch_step(G, S, step, grid);
        }
        MK_HIP(hipGetLastError());
        if (int r = read_counts(h)) return r;
        const uint32_t slot = step % (sssp ? kMsSlots : 3);
        const bool drained = h.scan[slot] ? h.active[slot] == 0
                                          : h.cnt[slot] == 0 && (h.large[slot] >> 32) == 0;
        if (h.overflow || drained) break;
        if (step > limit || (!sssp && step + 1 >= g->n + 2))
          return fail(MK_ERR_STATE, "multi-source traversal did not drain");
        group = std::min<uint32_t>(group * 2, 8);
      }
      if (h.overflow) {
        // the BFS log ran out of room: enlarge and run again
        if (int r = alloc_log(uint64_t(log_cap) * 4)) return r;
        continue;
      }
      MK_HIP(hipEventRecord(ev1, stream));
      MK_HIP(hipEventSynchronize(ev1));
      float t = 0.f;
      MK_HIP(hipEventElapsedTime(&t, ev0, ev1));
      if (ms) *ms = t;
      k = nsrc;
      last_steps = h.steps;
      last_edges = h.stat[0].edges;
      if (profiling_on())
        // BFS: 256 B per slab, 8 B per entry (the neighbour's seen mask);
        // SSSP: 256 B per slab, 4 B per (entry, active source) distance
        prof_add_bytes(sssp ? "k_mssp_step" : "k_msbfs_level",
                       256.0 * double(h.stat[0].slabs) +
                           (sssp ? 4.0 * double(h.stat[0].pairs) : 8.0 * double(h.stat[0].edges)));
      if (!sssp) {
        // levels 0..steps-1 are non-empty; seg[steps] is the log length
        uint32_t segs[1];
        MK_HIP(hipMemcpy(segs, seg + h.steps, 4, hipMemcpyDeviceToHost));
        log_total = segs[0];
      }
      return MK_OK;
    }
    return fail(MK_ERR_STATE, "multi-source BFS log kept overflowing");
  }

  int read(uint32_t slot, uint32_t *out) {
    if (session ? (slot >= 64 || !((admitted >> slot) & 1ull)) : slot >= k)
      return fail(MK_ERR_RANGE, session ? "mk_msq_read: slot not admitted in this session"
                                        : "mk_msq_read: slot not in the last run");
    MK_HIP(hipSetDevice(g->device));
    if (sssp) return read_words(out, g->n, g->device, stream, ColumnOf{dist, slot});
    if (int r = read_buf.ensure(size_t(g->n) * 4)) return r;
    if (session) {
      // the log so far: levels 0 .. step - 1 are written
      uint32_t total = 0;
      MK_HIP(hipMemcpyAsync(&total, seg + step, 4, hipMemcpyDeviceToHost, stream));
      MK_HIP(hipStreamSynchronize(stream));
      log_total = std::min(total, log_cap);
      last_steps = step;
    }
    fill_u32(read_buf.as<uint32_t>(), kInf, g->n, stream);
    if (log_total)
      k_msbfs_read<<<blocks_for_threads(log_total), kBlock, 0, stream>>>(
          view(), slot, log_total, last_steps + 1, read_buf.as<uint32_t>());
    return read_words(out, g->n, g->device, stream, WordsOf{read_buf.as<uint32_t>()});
  }
};

}  // namespace mk

struct mk_msq {
  mk::MultiSource m;
};

using namespace mk;

extern "C" {

int mk_msq_create(mk_graph *g, int sssp, mk_msq **out) {
  if (!out) return fail(MK_ERR_BAD_ARG, "mk_msq_create: out is NULL");
  *out = nullptr;
  if (!g) return fail(MK_ERR_BAD_ARG, "mk_msq_create: NULL graph");
  if (sssp && !g->weighted) return fail(MK_ERR_BAD_ARG, "multi-source SSSP needs a weighted graph");
  mk_msq *h = new mk_msq();
  int r = h->m.init(g, sssp != 0);
  if (r) {
    h->m.destroy();
    delete h;
    return r;
  }
  g->users++;
  *out = h;
  return MK_OK;
}

int mk_msq_destroy(mk_msq *q) {
  if (!q) return fail(MK_ERR_BAD_ARG, "mk_msq_destroy: NULL handle");
  q->m.g->users--;
  q->m.destroy();
  delete q;
  return MK_OK;
}

int mk_msq_run(mk_msq *q, const uint32_t *sources_host, uint32_t k, float *ms) {
  if (!q || (k && !sources_host)) return fail(MK_ERR_BAD_ARG, "mk_msq_run: NULL argument");
  if (k == 0 || k > 64) return fail(MK_ERR_BAD_ARG, "mk_msq_run: 1..64 sources");
  for (uint32_t i = 0; i < k; ++i)
    if (sources_host[i] >= q->m.g->n) return fail(MK_ERR_RANGE, "mk_msq_run: source >= n");
  if (int r = graph_settle(q->m.g)) return r;
  return q->m.run(sources_host, k, ms);
}

int mk_msq_open(mk_msq *q) {
  if (!q) return fail(MK_ERR_BAD_ARG, "mk_msq_open: NULL handle");
  if (int r = graph_settle(q->m.g)) return r;
  return q->m.open();
}

int mk_msq_admit(mk_msq *q, const uint32_t *sources_host, const uint32_t *slots_host, uint32_t k) {
  if (!q || (k && (!sources_host || !slots_host)))
    return fail(MK_ERR_BAD_ARG, "mk_msq_admit: NULL argument");
  if (k > 64) return fail(MK_ERR_BAD_ARG, "mk_msq_admit: at most 64 sources");
  return q->m.admit(sources_host, slots_host, k);
}

int mk_msq_launch(mk_msq *q, uint32_t steps) {
  if (!q) return fail(MK_ERR_BAD_ARG, "mk_msq_launch: NULL handle");
  return q->m.launch(steps);
}

int mk_msq_ready(mk_msq *q, int *ready) {
  if (!q || !ready) return fail(MK_ERR_BAD_ARG, "mk_msq_ready: NULL argument");
  MK_HIP(hipSetDevice(q->m.g->device));
  const hipError_t e = hipStreamQuery(q->m.stream);
  if (e == hipErrorNotReady) {
    *ready = 0;
    return MK_OK;
  }
  if (e != hipSuccess) return hip_fail(e, "mk_msq_ready");
  *ready = 1;
  return MK_OK;
}

int mk_msq_poll(mk_msq *q, uint64_t *active, uint32_t *steps) {
  if (!q || !active) return fail(MK_ERR_BAD_ARG, "mk_msq_poll: NULL argument");
  return q->m.poll(active, steps);
}

int mk_msq_read(mk_msq *q, uint32_t slot, uint32_t *dist_host) {
  if (!q || !dist_host) return fail(MK_ERR_BAD_ARG, "mk_msq_read: NULL argument");
  return q->m.read(slot, dist_host);
}

int mk_msq_last_stats(mk_msq *q, uint32_t *steps, uint64_t *edges) {
  if (!q) return fail(MK_ERR_BAD_ARG, "mk_msq_last_stats: NULL handle");
  if (steps) *steps = q->m.last_steps;
  if (edges) *edges = q->m.last_edges;
  return MK_OK;
}

}  // extern "C"
