// Triangle counting over an undirected graph stored in both directions.
//
// Reference: include/Algorithms/TC.cuh:9-41 and impl/TCImpl.cuh.  Static
// (:288-380) counts, for every directed edge (u, v) oriented from the lower
// degree end, the neighbours w of u found in adj[v] by a warp SearchEdge
// (TriangleCount_1, :149-214), and divides by 6 (:368).  Incremental
// (:431-497) and Decremental (:499-565) combine three counts over the batch
// graph in closed form.
//
// Method here (same counts):
//  - Static: vertices are ranked by (degree, id) and N+(x) holds the
//    neighbours of x ranked above x (|N+(x)| <= sqrt(2m)), as ranks, sorted.
//    Each triangle a < b < c is counted once, at b: as a c past b in N+(a),
//    for an a with b in N+(a), that is in N+(b) too.  Every vertex b has the
//    list of its (a, place of b in N+(a)); a wave puts N+(b) into LDS and
//    tests the tails of those N+(a) against it, so that every wedge is
//    looked at once (see "wedges" below).  Where the device memory for
//    these lists (16 bytes per undirected edge) is short, the N+ lists
//    alone (4 bytes) are built, a wave per vertex a puts N+(a) into an LDS
//    hash table and every N+(b) is streamed through it.
//  - Incremental / Decremental: the batch's changed undirected edges (the
//    entries the last insert / delete applied) go into a device hash set.
//    For each changed edge {u, v} the wave enumerates the neighbours w of the
//    cheaper end and tests the other end; a triangle found with j changed
//    edges among its three adds 6 / j, so each changed triangle sums to 6
//    over its j changed edges and the total / 6 is exact (no closed form over
//    separate counts).  For deletions the neighbourhoods are those before
//    the delete: current slabs plus the deleted edges (a CSR of the deleted
//    set built per call).
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <numeric>

#include "profile.hpp"
#include "slabhash.hpp"

namespace mk {

constexpr uint64_t kNoKey = ~0ull;
constexpr uint32_t kTcSlots = 64;

// rank(a) < rank(b) for (degree, id) ordering.
MK_DEV bool rank_lt(uint32_t da, uint32_t a, uint32_t db, uint32_t b) {
  return da < db || (da == db && a < b);
}

// Orders the wave's LDS accesses before and after it (the LDS unit takes a
// wave's accesses in order: no instruction, the compiler only).
MK_DEV void lds_settle() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

MK_DEV uint64_t edge_key(uint32_t a, uint32_t b) {
  return a < b ? (uint64_t(a) << 32) | b : (uint64_t(b) << 32) | a;
}
MK_DEV uint32_t key_slot(uint64_t k, uint32_t mask) {
  uint64_t h = k * 0x9E3779B97F4A7C15ull;
  return uint32_t(h >> 32) & mask;
}
// Insert into the open-addressing set; true if the key was not present.
MK_DEV bool set_insert(unsigned long long *tab, uint32_t mask, uint64_t k) {
  uint32_t h = key_slot(k, mask);
  for (;;) {
    const unsigned long long old = atomicCAS(tab + h, kNoKey, (unsigned long long)k);
    if (old == kNoKey) return true;
    if (old == k) return false;
    h = (h + 1) & mask;
  }
}
MK_DEV bool set_contains(const unsigned long long *tab, uint32_t mask, uint64_t k) {
  uint32_t h = key_slot(k, mask);
  for (;;) {
    const unsigned long long x = tab[h];
    if (x == k) return true;
    if (x == kNoKey) return false;
    h = (h + 1) & mask;
  }
}

MK_DEV void add_count(unsigned long long *slots, uint64_t v) {
  if (v) atomicAdd(&slots[blockIdx.x % kTcSlots], (unsigned long long)v);
}

// Static count over higher-ranked neighbour lists.  With vertices ranked by
// (degree, id) and N+(x) the neighbours of x ranked above x, every triangle
// a < b < c is counted once, at a, as an element of N+(a) \cap N+(b) for
// b in N+(a).  Pass 1 counts |N+(a)|, an exclusive scan places the lists,
// pass 2 writes them (compact, in HBM); the intersection kernel puts N+(a)
// (in chunks of kUpChunk) in an LDS hash table and streams each N+(b)
// through it with coalesced loads.

// Wave-collective walk of all slabs of vertex a (buckets loaded four at a
// time); for every live key x ranked above a calls f(up-ballot, x).
template <bool MAP, typename F>
MK_DEV void walk_up(const GraphView &G, uint32_t a, uint32_t da, uint32_t &slabs, F f) {
  const uint32_t lane = lane_id();
  const bool key_lane = (key_mask<MAP>() >> lane) & 1ull;
  const uint32_t b0 = G.bucket_off[a], b1 = G.bucket_off[a + 1];
  for (uint32_t bk = b0; bk < b1; bk += 4) {
    uint32_t x[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
      x[k] = bk + k < b1 ? G.heads[size_t(bk + k) * kSlabWords + lane] : kEmpty;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      if (bk + k >= b1) break;
      uint32_t v = x[k];
      for (;;) {
        ++slabs;
        const bool live = key_lane && v < kTomb;
        const uint32_t dv = live ? G.vdeg[v] : 0u;
        const bool up = live && rank_lt(da, a, dv, v);
        f(ballot(up), up, v);
        const uint32_t nx = read_lane(v, kNextLane);
        if (nx == kEmpty) break;
        v = slab_ptr(G.pool, nx)[lane];
      }
    }
  }
}

// Vertices are handed to waves kGrab at a time from a device counter: RMAT
// puts its heavy vertices at ids with many low zero bits, so a fixed
// grid stride (a power of two) would give them all to the same few waves.
constexpr uint32_t kGrab = 16;

// 64-bit so the counter cannot wrap past n while waves are still taking.
MK_DEV uint64_t grab(unsigned long long *next) {
  unsigned long long a0 = 0;
  if (lane_id() == 0) a0 = atomicAdd(next, (unsigned long long)kGrab);
  const uint32_t lo = read_lane(uint32_t(a0), 0), hi = read_lane(uint32_t(a0 >> 32), 0);
  return (uint64_t(hi) << 32) | lo;
}

template <bool MAP>
__global__ void __launch_bounds__(kBlock)
    k_tc_count_up(GraphView G, unsigned long long *K, unsigned long long *slab_count,
                  unsigned long long *next) {
  const uint32_t lane = lane_id();
  uint32_t slabs = 0;
  for (uint64_t a0 = grab(next); a0 < G.n; a0 = grab(next)) {
    const uint32_t a1 = uint32_t(min<uint64_t>(a0 + kGrab, G.n));
    for (uint32_t a = uint32_t(a0); a < a1; ++a) {
      const uint32_t da = G.vdeg[a];
      uint64_t k = 0;
      if (da) walk_up<MAP>(G, a, da, slabs, [&](uint64_t m, bool, uint32_t) { k += __popcll(m); });
      if (lane == 0) K[a] = k;
    }
  }
  if (lane == 0 && slabs) atomicAdd(slab_count, (unsigned long long)slabs);
}

template <bool MAP>
__global__ void __launch_bounds__(kBlock)
    k_tc_fill_up(GraphView G, const unsigned long long *off, uint32_t *up,
                 unsigned long long *slab_count, unsigned long long *next) {
  uint32_t slabs = 0;
  for (uint64_t a0 = grab(next); a0 < G.n; a0 = grab(next))
  for (uint32_t a = uint32_t(a0); a < uint32_t(min<uint64_t>(a0 + kGrab, G.n)); ++a) {
    const uint32_t da = G.vdeg[a];
    if (!da) continue;
    uint64_t pos = off[a];
    walk_up<MAP>(G, a, da, slabs, [&](uint64_t m, bool mine, uint32_t v) {
      if (mine) up[pos + lanes_below(m)] = v;
      pos += __popcll(m);
    });
  }
  if (lane_id() == 0 && slabs) atomicAdd(slab_count, (unsigned long long)slabs);
}

constexpr uint32_t kUpChunk = 1024;     // N+(a) keys per LDS table fill
constexpr uint32_t kHashSlots = 2048;   // LDS hash slots per wave (load <= 1/2)

MK_DEV uint32_t lds_slot(uint32_t x) { return (x * 2654435761u) >> (32 - 11); }

__global__ void __launch_bounds__(kBlock)
    k_tc_intersect(const unsigned long long *off, const uint32_t *up, uint32_t n,
                   unsigned long long *slots, unsigned long long *streamed,
                   unsigned long long *next) {
  static_assert(kHashSlots == 1u << 11, "lds_slot assumes 2048 slots");
  const uint32_t lane = lane_id();
  __shared__ uint32_t table[kBlock / 64][kHashSlots];
  uint32_t *h = table[threadIdx.x >> 6];
  uint64_t count = 0, reads = 0;
  for (uint64_t a0 = grab(next); a0 < n; a0 = grab(next))
  for (uint32_t a = uint32_t(a0); a < uint32_t(min<uint64_t>(a0 + kGrab, n)); ++a) {
    const uint64_t oa = off[a];
    const uint32_t Ka = uint32_t(off[a + 1] - oa);
    if (Ka < 2) continue;
    for (uint32_t c0 = 0; c0 < Ka; c0 += kUpChunk) {
      const uint32_t cn = min(kUpChunk, Ka - c0);
      for (uint32_t i = lane; i < kHashSlots; i += 64) h[i] = kEmpty;
      __builtin_amdgcn_wave_barrier();
      for (uint32_t i = lane; i < cn; i += 64) {
        const uint32_t x = up[oa + c0 + i];
        uint32_t sl = lds_slot(x);
        while (atomicCAS(h + sl, kEmpty, x) != kEmpty) sl = (sl + 1) & (kHashSlots - 1);
      }
      __builtin_amdgcn_wave_barrier();
      // every b in N+(a): count N+(b) elements in this chunk of N+(a); the
      // next b's list bounds load while the current list streams, four
      // 64-element rows at a time
      uint32_t bn = up[oa];
      uint64_t obn = off[bn], oen = off[bn + 1];
      for (uint32_t i = 0; i < Ka; ++i) {
        const uint64_t ob = obn;
        const uint32_t Kb = uint32_t(oen - obn);
        if (i + 1 < Ka) {
          bn = up[oa + i + 1];
          obn = off[bn];
          oen = off[bn + 1];
        }
        reads += Kb;
        for (uint32_t j0 = 0; j0 < Kb; j0 += 256) {
          uint32_t c[4];
#pragma unroll
          for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t j = j0 + k * 64 + lane;
            c[k] = j < Kb ? up[ob + j] : kEmpty;  // ids are < kEmpty
          }
#pragma unroll
          for (uint32_t k = 0; k < 4; ++k) {
            if (c[k] == kEmpty) continue;
            uint32_t sl = lds_slot(c[k]);
            for (;;) {
              const uint32_t e = h[sl];
              if (e == c[k]) {
                ++count;
                break;
              }
              if (e == kEmpty) break;
              sl = (sl + 1) & (kHashSlots - 1);
            }
          }
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  count = wave_sum_u64(count);
  if (lane == 0) {
    add_count(slots, count);
    if (reads) atomicAdd(streamed, (unsigned long long)reads);
  }
}

// ---------------------------------------------------------------- wedges
// The static count over sorted lists of ranks.  RMAT-20 (15.7M undirected
// edges): the tails tested are 1.23e9 elements, where streaming every N+(b)
// against N+(a) reads 4.42e9.
constexpr uint32_t kTableWords = 1024;  // LDS words per wave: bitmap or hash table
constexpr uint32_t kTopRanks = kTableWords * 32;  // highest ranks a bitmap covers exactly
constexpr uint32_t kUnit = 64;          // list entries per unit of k_tc_wedges
constexpr uint32_t kTakers = 16;         // unit counters
constexpr uint64_t kSmallTotal = 1u << 16;
constexpr uint32_t kSortRow = 1024;     // row elements staged in LDS at a time
constexpr uint32_t kTail = 8;           // lanes per tail
constexpr uint32_t kRounds = 4;         // elements a lane takes at a time

__global__ void k_tc_iota(uint32_t *p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = i;
}

// rank[order[i]] = i; row i (a rank) starts with room for its whole degree.
__global__ void k_tc_rank(const uint32_t *order, const uint32_t *sdeg, uint32_t n, uint32_t *rank,
                          unsigned long long *deg) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  rank[order[i]] = i;
  deg[i] = sdeg[i];
}

// One pass over the slabs, an 8-lane group per bucket: the ranks above the
// owner's, appended to the owner's row (`cursor`: one atomic per slab).
// Rows have room for the whole degree, so nothing is counted first.  Bound
// by the rank gathers (one per key, from an array of 4 bytes a vertex).
template <bool MAP>
__global__ void __launch_bounds__(kBlock)
    k_tc_rows(GraphView G, const uint32_t *rank, const unsigned long long *row0, uint32_t *len,
              uint32_t *raw, unsigned long long *slab_count) {
  const uint32_t gl = group_lane();
  const uint64_t g0 = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) / kGroupLanes;
  const uint64_t NG = uint64_t(gridDim.x) * blockDim.x / kGroupLanes;
  uint32_t slabs = 0;
  for (uint64_t b = g0; b < G.total_buckets; b += NG) {
    const uint32_t u = G.bucket_owner[b];
    if (G.vdeg[u] == 0) continue;
    const uint32_t r = rank[u];
    const uint32_t *slab = G.heads + b * kSlabWords;
    for (;;) {
      ++slabs;
      uint32_t x[kWordsPerLane], rx[kWordsPerLane];
      load_words(slab + kWordsPerLane * gl, x);
      uint32_t c = 0;
#pragma unroll
      for (uint32_t k = 0; k < kWordsPerLane; ++k)
        rx[k] = key_word<MAP>(kWordsPerLane * gl + k) && x[k] < kTomb ? rank[x[k]] : 0u;
#pragma unroll
      for (uint32_t k = 0; k < kWordsPerLane; ++k) c += rx[k] > r ? 1u : 0u;
      uint32_t pre = c;  // inclusive over the group
#pragma unroll
      for (uint32_t o = 1; o < kGroupLanes; o <<= 1) {
        const uint32_t y = uint32_t(__shfl_up(int(pre), o, int(kGroupLanes)));
        if (gl >= o) pre += y;
      }
      const uint32_t sum = group_read(pre, kGroupLanes - 1);
      if (sum) {
        uint32_t at = 0;
        if (gl == 0) at = atomicAdd(len + r, sum);
        unsigned long long pos = row0[r] + group_read(at, 0) + (pre - c);
#pragma unroll
        for (uint32_t k = 0; k < kWordsPerLane; ++k)
          if (rx[k] > r) raw[pos++] = rx[k];
      }
      const uint32_t nx = group_read(x[kWordsPerLane - 1], kGroupLanes - 1);
      if (nx == kEmpty) break;
      slab = slab_ptr(G.pool, nx);
    }
  }
  slabs = wave_sum_u32(gl == 0 ? slabs : 0u);
  if (lane_id() == 0 && slabs) atomicAdd(slab_count, (unsigned long long)slabs);
}

// Where vertex b's list counter lies: neighbouring ranks, all hubs at the
// top, are kSpread columns apart, so that their counters share no line
// (atomics on one line follow one another: RMAT-20's counts took 2.6 ms in
// rank order).
constexpr uint32_t kSpread = 1024;
__host__ __device__ inline uint32_t spread_rows(uint32_t n) { return (n + kSpread - 1) / kSpread; }
MK_DEV uint32_t spread_index(uint32_t b, uint32_t n) {
  return (b % kSpread) * spread_rows(n) + b / kSpread;
}

// Row (or spread list) lengths as 64-bit values with a zero behind them.
__global__ void k_tc_widen(const uint32_t *len, uint32_t n, bool spread, unsigned long long *out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i <= n) out[i] = i < n ? len[spread ? spread_index(i, n) : i] : 0ull;
}

// Sort every row (ranks are distinct: an element's place is the number of
// smaller ones) into `up`, and give every element b but a row's last, whose
// tail is empty, its place in b's list: slot[e] = entries of b so far
// (kEmpty: none, also when N+(b) is empty).  A wave takes 64 rows: single
// elements lane by lane, rows of up to 64 in registers, longer ones staged
// in LDS kSortRow at a time.
MK_DEV uint32_t tc_slot(uint32_t b, bool tail, const uint32_t *len, uint32_t *ndown, uint32_t n) {
  return tail && len[b] ? atomicAdd(ndown + spread_index(b, n), 1u) : kEmpty;
}
__global__ void __launch_bounds__(kBlock)
    k_tc_sort(const unsigned long long *row0, const uint32_t *len, const unsigned long long *off,
              const uint32_t *raw, uint32_t n, uint32_t *up, uint32_t *slot, uint32_t *ndown) {
  __shared__ uint32_t stage[kBlock / 64][kSortRow];
  const uint32_t lane = lane_id();
  uint32_t *st = stage[threadIdx.x >> 6];
  const uint64_t gw = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const uint64_t W = (uint64_t(gridDim.x) * blockDim.x) >> 6;
  for (uint64_t r0 = gw; r0 * 64 < n; r0 += W) {
    // lane i: row i * ceil(n / 64) + r0, so that a wave's rows are spread
    // over the ranks (long rows are neighbours)
    const uint64_t r = uint64_t(lane) * ((uint64_t(n) + 63) / 64) + r0;
    const bool mine = r < n && r0 < (uint64_t(n) + 63) / 64;
    const uint32_t K = mine ? len[r] : 0u;
    const unsigned long long src = mine ? row0[r] : 0ull, dst = mine ? off[r] : 0ull;
    if (K == 1) {
      up[dst] = raw[src];
      slot[dst] = kEmpty;
    }
    uint64_t m = ballot(K > 1);
    while (m) {
      const uint32_t j = ffs64(m);
      m &= m - 1;
      const uint32_t k = read_lane(K, j);
      const uint32_t *in = raw + (uint64_t(read_lane(uint32_t(src >> 32), j)) << 32 |
                                  read_lane(uint32_t(src), j));
      const unsigned long long o = uint64_t(read_lane(uint32_t(dst >> 32), j)) << 32 |
                                   read_lane(uint32_t(dst), j);
      if (k <= 64) {
        const uint32_t x = lane < k ? in[lane] : kEmpty;
        uint32_t at = 0;
        for (uint32_t i = 0; i < k; ++i) at += read_lane(x, i) < x ? 1u : 0u;
        if (lane < k) {
          up[o + at] = x;
          slot[o + at] = tc_slot(x, at + 1 < k, len, ndown, n);
        }
        continue;
      }
      for (uint32_t c0 = 0; c0 < k; c0 += 64) {
        const uint32_t x = c0 + lane < k ? in[c0 + lane] : kEmpty;
        uint32_t at = 0;
        for (uint32_t t0 = 0; t0 < k; t0 += kSortRow) {
          const uint32_t tn = min(kSortRow, k - t0);
          if (c0 == 0 || k > kSortRow) {  // one tile: staged once
            lds_settle();
            for (uint32_t i = lane; i < (tn + 3) / 4 * 4; i += 64)
              st[i] = i < tn ? in[t0 + i] : kEmpty;
            lds_settle();
          }
          for (uint32_t i = 0; i < tn; i += 4) {
            const uint4 y = *reinterpret_cast<const uint4 *>(st + i);
            at += (y.x < x ? 1u : 0u) + (y.y < x ? 1u : 0u) + (y.z < x ? 1u : 0u) +
                  (y.w < x ? 1u : 0u);
          }
        }
        if (c0 + lane < k) {
          up[o + at] = x;
          slot[o + at] = tc_slot(x, at + 1 < k, len, ndown, n);
        }
      }
      lds_settle();
    }
  }
}

// Entry of b's list: the tail of a row past b, (first element << 24) | length.
// Rows shorter than 2^24 (their square is at most 2 m).  Eight rows to a
// wave: neighbouring ranks' rows are long together (64 to a wave left the
// last waves running for 0.9 ms on RMAT-20).
constexpr uint32_t kDownRows = 8;
__global__ void __launch_bounds__(kBlock)
    k_tc_down(const uint32_t *len, const unsigned long long *off, const uint32_t *up,
              const uint32_t *slot, const unsigned long long *doff, uint32_t n,
              unsigned long long *down) {
  const uint32_t lane = lane_id();
  const uint64_t gw = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const uint64_t W = (uint64_t(gridDim.x) * blockDim.x) >> 6;
  for (uint64_t r0 = gw * kDownRows; r0 < n; r0 += W * kDownRows) {
    // the rows' elements together, 64 at a time
    const uint32_t K = lane < kDownRows && r0 + lane < n ? len[r0 + lane] : 0u;
    uint32_t incl = K;
#pragma unroll
    for (uint32_t o = 1; o < kDownRows; o <<= 1) {
      const uint32_t y = uint32_t(__shfl_up(int(incl), o, 64));
      if (lane >= o) incl += y;
    }
    const uint32_t total = read_lane(incl, kDownRows - 1);
    const unsigned long long base = off[r0];
    for (uint32_t e = lane; e < total; e += 64) {
      uint32_t end = total;  // the end of e's row
#pragma unroll
      for (uint32_t k = kDownRows - 1; k > 0; --k) {
        const uint32_t x = read_lane(incl, k - 1);
        if (e < x) end = x;
      }
      const uint32_t s = slot[base + e];
      if (s != kEmpty) down[doff[up[base + e]] + s] = ((base + e + 1) << 24) | (end - e - 1);
    }
  }
}

// The vertex whose list holds the first entry of every unit.
__global__ void k_tc_units(const unsigned long long *doff, uint32_t n, uint32_t *unit_b) {
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= n) return;
  for (unsigned long long u = (doff[b] + kUnit - 1) / kUnit; u * kUnit < doff[b + 1]; ++u)
    unit_b[u] = b;
}

MK_DEV uint32_t table_slot(uint32_t x) {
  static_assert(kTableWords == 1u << 10, "ten hash bits");
  return (x * 2654435761u) >> (32 - 10);
}

// The wedges of one run of entries [s, e) of vertex b against N+(b) in the
// wave's table.  Each 8-lane group takes every eighth entry, 32 elements of
// its tail at a time, the next 32 in flight; groups go on to their next
// entry independently.  BITS: exact bitmap of the ranks from `top` on; else an
// open-addressing hash table.
template <bool BITS>
MK_DEV void tc_tails(const uint32_t *tab, uint32_t top, const unsigned long long *down,
                     unsigned long long s, unsigned long long e, const uint32_t *up,
                     uint64_t &count) {
  const uint32_t gl = lane_id() & (kTail - 1);
  unsigned long long i = s + lane_id() / kTail;
  unsigned long long ent = i < e ? down[i] : 0ull;
  i += 64 / kTail;
  unsigned long long nxt = i < e ? down[i] : 0ull;
  unsigned long long p = ent >> 24, end = p + (ent & 0xFFFFFFull);
  uint32_t hits = 0;
  uint32_t c[kRounds], d[kRounds];  // this round's elements and the next one's, in flight
#pragma unroll
  for (uint32_t k = 0; k < kRounds; ++k) {
    const unsigned long long q = p + k * kTail + gl;
    d[k] = q < end ? up[q] : kEmpty;
  }
  bool more = ballot(p < end) != 0;
  while (more) {
    p += kRounds * kTail;
    if (p >= end) {  // the group's next entry (0: none, an empty tail)
      p = nxt >> 24;
      end = p + (nxt & 0xFFFFFFull);
      i += 64 / kTail;
      nxt = i < e ? down[i] : 0ull;
    }
    more = ballot(p < end) != 0;
#pragma unroll
    for (uint32_t k = 0; k < kRounds; ++k) {
      c[k] = d[k];
      const unsigned long long q = p + k * kTail + gl;
      d[k] = q < end ? up[q] : kEmpty;
    }
#pragma unroll
    for (uint32_t k = 0; k < kRounds; ++k) {
      if (c[k] == kEmpty) continue;
      if (BITS) {
        const uint32_t x = c[k] - top;
        hits += (tab[x >> 5] >> (x & 31u)) & 1u;
      } else {
        uint32_t sl = table_slot(c[k]);
        for (;;) {
          const uint32_t t = tab[sl];
          if (t == c[k]) {
            ++hits;
            break;
          }
          if (t == kEmpty) break;
          sl = (sl + 1) & (kTableWords - 1);
        }
      }
    }
  }
  count += hits;
}

// The wedge count: a wave per unit of kUnit consecutive list entries (units
// in a permuted order: neighbours cost alike), vertex after vertex of the
// unit.  N+(b) goes into the wave's table: for the kTopRanks highest ranks
// a bitmap (every element is ranked above b, so the table is exact; one LDS
// read a test), below them a hash table of up to kTableWords / 2 elements at
// a time.  Bound by the latency of the tails' loads, so the table is small
// enough for 32 waves a CU: RMAT-20's 1.23e9 tests take 1.10 ms, 1.83 ms at
// 2048 words (20 waves a CU); units of 256 entries took as long there, but
// 2.4x at RMAT-17, whose last units ran alone; 16 lanes a tail 1.17 ms.
__global__ void __launch_bounds__(kBlock)
    k_tc_wedges(const uint32_t *len, const unsigned long long *off, const uint32_t *up,
                const unsigned long long *doff, const unsigned long long *down,
                const uint32_t *unit_b, uint32_t n, uint64_t entries, uint64_t units,
                uint64_t stride, unsigned long long *next, unsigned long long *slots) {
  if (entries == 0) {  // the host did not wait for them
    entries = doff[n];
    units = (entries + kUnit - 1) / kUnit;
    stride = 1;
  }
  __shared__ uint32_t table[kBlock / 64][kTableWords];
  uint32_t *tab = table[threadIdx.x >> 6];
  const uint32_t lane = lane_id();
  const uint64_t gw = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const uint32_t top = n > kTopRanks ? n - kTopRanks : 0u;
  uint64_t count = 0;
  // waves take units from kTakers counters (a line each) that share the
  // units out between them: one counter would hand out a unit every 11 ns
  const uint32_t taker = uint32_t(gw % kTakers);
  for (;;) {
    unsigned long long t = 0;
    if (lane == 0) t = atomicAdd(next + taker * 16, 1ull);
    const uint64_t k =
        (uint64_t(read_lane(uint32_t(t >> 32), 0)) << 32 | read_lane(uint32_t(t), 0)) * kTakers +
        taker;
    if (k >= units) break;
    const uint64_t p0 = (k * stride % units) * kUnit, p1 = min(p0 + kUnit, entries);
    for (uint32_t b0 = unit_b[p0 / kUnit]; b0 < n; b0 += 64) {
      // 64 vertices' lists at once: those with entries in this unit
      const uint32_t bl = b0 + lane;
      const unsigned long long d0 = bl < n ? doff[bl] : entries;
      const unsigned long long d1 = bl < n ? doff[bl + 1] : entries;
      uint64_t m = ballot(d0 < d1 && d0 < p1 && d1 > p0);
      const bool last = ballot(d1 >= p1) != 0;
      while (m) {
        const uint32_t j = ffs64(m);
        m &= m - 1;
        const uint32_t b = b0 + j;
        const unsigned long long s = max<uint64_t>(doff[b], p0), e = min<uint64_t>(doff[b + 1], p1);
        const uint32_t K = len[b];
        const uint32_t *row = up + off[b];
        if (b >= top) {
          lds_settle();
          for (uint32_t i = lane * 4; i < kTableWords; i += 256)
            *reinterpret_cast<uint4 *>(tab + i) = make_uint4(0u, 0u, 0u, 0u);
          lds_settle();
          for (uint32_t i = lane; i < K; i += 64) {
            const uint32_t x = row[i] - top;
            atomicOr(tab + (x >> 5), 1u << (x & 31u));
          }
          lds_settle();
          tc_tails<true>(tab, top, down, s, e, up, count);
        } else {
          for (uint32_t c0 = 0; c0 < K; c0 += kTableWords / 2) {
            const uint32_t cn = min(kTableWords / 2, K - c0);
            lds_settle();
            for (uint32_t i = lane * 4; i < kTableWords; i += 256)
              *reinterpret_cast<uint4 *>(tab + i) = make_uint4(kEmpty, kEmpty, kEmpty, kEmpty);
            lds_settle();
            for (uint32_t i = lane; i < cn; i += 64) {
              const uint32_t x = row[c0 + i];
              uint32_t sl = table_slot(x);
              while (atomicCAS(tab + sl, kEmpty, x) != kEmpty) sl = (sl + 1) & (kTableWords - 1);
            }
            lds_settle();
            tc_tails<false>(tab, 0u, down, s, e, up, count);
          }
        }
      }
      if (last) break;
    }
  }
  count = wave_sum_u64(count);
  if (lane == 0) add_count(slots, count);
}

// The end of a changed edge that is enumerated (x, fewer live neighbours) and
// the one that is tested (y).
MK_DEV uint2 tc_ends(const GraphView &G, uint2 uv) {
  return G.vdeg[uv.x] > G.vdeg[uv.y] ? make_uint2(uv.y, uv.x) : uv;
}

// Canonical changed edges of a batch: entries with status == APPLIED (or all
// non-loop entries when status is NULL) enter the set; the first entry of
// each undirected edge appends it to `owned` and adds the buckets of its
// enumerated end to *n_items.
__global__ void __launch_bounds__(kBlock)
    k_tc_collect(GraphView G, const uint32_t *src, const uint32_t *dst, const uint8_t *status, uint32_t n,
                 uint32_t nv, unsigned long long *tab, uint32_t mask, uint2 *owned,
                 uint32_t *n_owned, unsigned long long *n_items) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  bool mine = false;
  uint32_t u = 0, v = 0;
  if (i < n) {
    u = src[i];
    v = dst[i];
    const bool ok = u != v && u < nv && v < nv && (!status || status[i] == MK_EDGE_APPLIED);
    if (ok) mine = set_insert(tab, mask, edge_key(u, v));
  }
  const uint64_t m = ballot(mine);
  if (m) {
    uint32_t base = 0;
    const uint32_t leader = ffs64(m);
    if (lane_id() == leader) base = atomicAdd(n_owned, uint32_t(__popcll(m)));
    base = read_lane(base, leader);
    if (mine) owned[base + lanes_below(m)] = make_uint2(min(u, v), max(u, v));
    uint32_t nb = 0;
    if (mine) {
      const uint32_t x = tc_ends(G, make_uint2(min(u, v), max(u, v))).x;
      nb = G.bucket_off[x + 1] - G.bucket_off[x];
    }
    const uint64_t sum = wave_sum_u64(nb);
    if (lane_id() == leader) atomicAdd(n_items, (unsigned long long)sum);
  }
}

// Most work items at a time (32 MB): a batch that has more, hub-to-hub edges
// mostly, is worked in passes over windows of them.
constexpr uint64_t kMaxItems = 1ull << 22;

// Work items of the changed edges: (edge, bucket of its enumerated end), the
// edge's items side by side; one claim on *next per wave.  With `start`
// (batches of several windows) the claims, made by window 0, stay there, and
// only the items lo, lo + 1, ... below hi are written.
__global__ void __launch_bounds__(kBlock)
    k_tc_items(GraphView G, const uint2 *owned, uint32_t n_owned, uint2 *items,
               unsigned long long *next, unsigned long long *start, uint64_t lo, uint64_t hi) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lane = lane_id();
  uint32_t nb = 0;
  if (i < n_owned) {
    const uint32_t x = tc_ends(G, owned[i]).x;
    nb = G.bucket_off[x + 1] - G.bucket_off[x];
  }
  uint64_t incl = nb;
#pragma unroll
  for (uint32_t o = 1; o < 64; o <<= 1) {
    const uint64_t y = (uint64_t(uint32_t(__shfl_up(int(incl >> 32), o, 64))) << 32) |
                       uint32_t(__shfl_up(int(uint32_t(incl)), o, 64));
    if (lane >= o) incl += y;
  }
  unsigned long long base = 0;
  if (lo == 0) {
    if (lane == 63) base = atomicAdd(next, (unsigned long long)incl);
    base = (uint64_t(read_lane(uint32_t(base >> 32), 63)) << 32) | read_lane(uint32_t(base), 63);
    base += incl - nb;
    if (start && nb) start[i] = base;
  } else if (nb) {
    base = start[i];
  }
  const uint32_t j0 = base < lo ? uint32_t(min<uint64_t>(lo - base, nb)) : 0u;
  const uint32_t j1 = base < hi ? uint32_t(min<uint64_t>(hi - base, nb)) : 0u;
  for (uint32_t j = j0; j < j1; ++j) items[base + j - lo] = make_uint2(i, j);
}

// Weight of a triangle with j changed edges: 6 / j.
MK_DEV uint32_t six_over(uint32_t j) { return j == 1 ? 6u : (j == 2 ? 3u : 2u); }

// Test the keys c of the lanes with `act` against vertex y's adjacency: the
// keys are packed into LDS and each 8-lane group tests two at a time, so
// that sixteen of y's slabs are in flight per wave (a wave-wide walk had one:
// a key and its slab after the other).  Returns whether this lane's key is
// there.  Wave-collective.
template <bool MAP>
MK_DEV bool tc_test_keys(const GraphView &G, uint32_t y, bool act, uint32_t c, uint32_t *lds,
                         uint32_t &slabs) {
  const uint32_t gl = group_lane(), grp = lane_id() / kGroupLanes;
  const uint64_t m = ballot(act);
  const uint32_t n = uint32_t(__popcll(m));
  lds_settle();
  if (act) lds[lanes_below(m)] = c;
  lds_settle();
  const uint32_t off = G.bucket_off[y], nb = G.bucket_off[y + 1] - off;
  for (uint32_t k0 = 0; k0 < n; k0 += 2 * kGroupsPerWave) {
    uint32_t key[2], v[2][kWordsPerLane];
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) {
      const uint32_t k = k0 + q * kGroupsPerWave + grp;
      key[q] = k < n ? lds[k] : kEmpty;
      if (key[q] != kEmpty)
        load_words(G.heads + size_t(off + bucket_in(key[q], nb)) * kSlabWords + kWordsPerLane * gl,
                   v[q]);
    }
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) {
      if (key[q] == kEmpty) continue;
      bool found = false;
      for (;;) {
        if (gl == 0) ++slabs;
        bool hit = false;
#pragma unroll
        for (uint32_t j = 0; j < kWordsPerLane; ++j)
          hit |= key_word<MAP>(kWordsPerLane * gl + j) && v[q][j] == key[q];
        found = group_bits(ballot(hit)) != 0u;
        const uint32_t nx = group_read(v[q][kWordsPerLane - 1], kGroupLanes - 1);
        if (found || nx == kEmpty) break;
        load_words(slab_ptr(G.pool, nx) + kWordsPerLane * gl, v[q]);
      }
      if (gl == 0) lds[k0 + q * kGroupsPerWave + grp] = found ? 1u : 0u;
    }
  }
  lds_settle();
  return act && lds[lanes_below(m)] != 0u;
}

// Triangles through each inserted edge {u, v} (graph already updated): w
// over adj[x] of the lower-degree end x, tested in adj[y]; a wave per item
// (edge, bucket of x), so that a hub's buckets are spread over the device.
// Bound by the latency of y's slabs.  RMAT-18, 50k edges of the same
// distribution: 0.38 ms; 1.64 ms with a wave per edge (the hub edges'
// waves ran last, alone) that tested a key after the other.
template <bool MAP>
__global__ void __launch_bounds__(kBlock)
    k_tc_inserted(GraphView G, const uint2 *owned, const uint2 *items, uint64_t n_items,
                  const unsigned long long *tab, uint32_t mask, unsigned long long *slots,
                  unsigned long long *slab_count) {
  __shared__ uint32_t keys[kBlock / 64][64];
  uint32_t *lds = keys[threadIdx.x >> 6];
  const uint32_t lane = lane_id();
  const uint64_t gw = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const uint64_t W = (uint64_t(gridDim.x) * blockDim.x) >> 6;
  const bool key_lane = (key_mask<MAP>() >> lane) & 1ull;
  uint64_t count = 0;
  uint32_t slabs = 0;
  for (uint64_t t = gw; t < n_items; t += W) {
    const uint2 it = items[t];
    const uint2 xy = tc_ends(G, owned[it.x]);
    const uint32_t x = xy.x, y = xy.y;
    const uint32_t *slab = G.heads + size_t(G.bucket_off[x] + it.y) * kSlabWords;
    for (;;) {
      const uint32_t w = slab[lane];
      if (lane == 0) ++slabs;
      const bool act = key_lane && w < kTomb && w != y;
      if (tc_test_keys<MAP>(G, y, act, w, lds, slabs))
        count += six_over(1u + (set_contains(tab, mask, edge_key(x, w)) ? 1u : 0u) +
                          (set_contains(tab, mask, edge_key(y, w)) ? 1u : 0u));
      const uint32_t nx = read_lane(w, kNextLane);
      if (nx == kEmpty) break;
      slab = slab_ptr(G.pool, nx);
    }
  }
  count = wave_sum_u64(count);
  slabs = wave_sum_u32(slabs);
  if (lane == 0) {
    add_count(slots, count);
    if (slabs) atomicAdd(slab_count, (unsigned long long)slabs);
  }
}

// Degree of every vertex in the deleted set (both ends of each edge).
__global__ void k_tc_dcount(const uint2 *owned, uint32_t n_owned, uint32_t *ddeg) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_owned) return;
  atomicAdd(ddeg + owned[i].x, 1u);
  atomicAdd(ddeg + owned[i].y, 1u);
}

__global__ void k_tc_dfill(const uint2 *owned, uint32_t n_owned, const uint32_t *doff,
                           uint32_t *cursor, uint32_t *dlist) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_owned) return;
  const uint2 e = owned[i];
  dlist[doff[e.x] + atomicAdd(cursor + e.x, 1u)] = e.y;
  dlist[doff[e.y] + atomicAdd(cursor + e.y, 1u)] = e.x;
}

// Triangles of the graph before the delete through each deleted edge
// {u, v}: w over (current adj[x]) + (deleted neighbours of x), tested
// against (current adj[y]) + (deleted neighbours of y, via the set).  Items
// as in k_tc_inserted; x's deleted neighbours are shared out over its items
// 64 at a time.  RMAT-18, 50k edges: 1.62 -> 0.56 ms.
template <bool MAP>
__global__ void __launch_bounds__(kBlock)
    k_tc_deleted(GraphView G, const uint2 *owned, const uint2 *items, uint64_t n_items,
                 const unsigned long long *tab, uint32_t mask, const uint32_t *doff,
                 const uint32_t *dlist, unsigned long long *slots, unsigned long long *slab_count) {
  __shared__ uint32_t keys[kBlock / 64][64];
  uint32_t *lds = keys[threadIdx.x >> 6];
  const uint32_t lane = lane_id();
  const uint64_t gw = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const uint64_t W = (uint64_t(gridDim.x) * blockDim.x) >> 6;
  const bool key_lane = (key_mask<MAP>() >> lane) & 1ull;
  uint64_t count = 0;
  uint32_t slabs = 0;
  for (uint64_t t = gw; t < n_items; t += W) {
    const uint2 it = items[t];
    const uint2 xy = tc_ends(G, owned[it.x]);
    const uint32_t x = xy.x, y = xy.y;
    // the changed edges of triangle {x, y, w}: {x, y}, {x, w} in part (b),
    // and {y, w} if it was deleted (then it is not in adj[y] now)
    auto tally = [&](bool act, uint32_t w, uint32_t changed) {
      const bool gone = act && set_contains(tab, mask, edge_key(y, w));
      const bool found = tc_test_keys<MAP>(G, y, act, w, lds, slabs);
      if (found || gone) count += six_over(changed + (gone ? 1u : 0u));
    };
    // (a) w in the current adjacency of x: {x, w} is not deleted
    const uint32_t b0 = G.bucket_off[x], nb = G.bucket_off[x + 1] - b0;
    const uint32_t *slab = G.heads + size_t(b0 + it.y) * kSlabWords;
    for (;;) {
      const uint32_t w = slab[lane];
      if (lane == 0) ++slabs;
      tally(key_lane && w < kTomb && w != y, w, 1u);
      const uint32_t nx = read_lane(w, kNextLane);
      if (nx == kEmpty) break;
      slab = slab_ptr(G.pool, nx);
    }
    // (b) w a deleted neighbour of x: {x, w} is deleted
    const uint32_t d0 = doff[x], d1 = doff[x + 1];
    for (uint64_t j0 = d0 + uint64_t(it.y) * 64; j0 < d1; j0 += uint64_t(nb) * 64) {
      const uint64_t j = j0 + lane;
      const uint32_t w = j < d1 ? dlist[j] : y;
      tally(w != y, w, 2u);
    }
  }
  count = wave_sum_u64(count);
  slabs = wave_sum_u32(slabs);
  if (lane == 0) {
    add_count(slots, count);
    if (slab_count && slabs) atomicAdd(slab_count, (unsigned long long)slabs);
  }
}

struct TC {
  mk_graph *g = nullptr;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  // kTcSlots counts, then the slab counter and the streamed-elements counter
  unsigned long long *slots = nullptr;
  uint32_t *n_owned = nullptr;  // [0] changed edges, [2..3] their items, [4..5] items written
  DevBuf tab, owned, ddeg, doff, cursor, dlist, scan_tmp, kup, koff, uplist, grabs;
  uint32_t word_seq = 0;        // of read_word
  DevBuf items, item_start;
  DevBuf ranks, rows, raw, slot, units;  // static count over sorted rows
  HostBuf host;
  unsigned long long count = 0;
  uint64_t last_slabs = 0, last_streamed = 0;
  int max_waves = 0;

  int init(mk_graph *graph) {
    g = graph;
    MK_HIP(hipSetDevice(g->device));
    MK_HIP(hipStreamCreate(&stream));
    loop_stream_add(g->device, stream, 1);
    MK_HIP(hipEventCreate(&ev0));
    MK_HIP(hipEventCreate(&ev1));
    MK_HIP(hipMalloc(&slots, (kTcSlots + 2) * 8));
    MK_HIP(hipMalloc(&n_owned, 32));
    if (int r = host.ensure((kTcSlots + 4) * 8)) return r;
    max_waves = grid_waves(g->device);
    return MK_OK;
  }

  void destroy() {
    (void)hipSetDevice(g->device);
    if (stream) (void)hipStreamSynchronize(stream);
    (void)hipFree(slots);
    (void)hipFree(n_owned);
    for (DevBuf *b :
         {&tab, &owned, &ddeg, &doff, &cursor, &dlist, &scan_tmp, &kup, &koff, &uplist, &grabs,
          &items, &item_start, &ranks, &rows, &raw, &slot, &units})
      b->release();
    host.release();
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) {
      loop_stream_add(g->device, stream, -1);
      (void)hipStreamDestroy(stream);
    }
  }

  int start() {
    MK_HIP(hipSetDevice(g->device));
    MK_HIP(hipEventRecord(ev0, stream));
    fill_u64(reinterpret_cast<uint64_t *>(slots), 0ull, kTcSlots + 2, stream);
    return MK_OK;
  }

  // Sum of the count slots; also ends timing.
  int finish(uint64_t &total, float *ms) {
    MK_HIP(hipGetLastError());
    MK_HIP(hipMemcpyAsync(host.ptr, slots, (kTcSlots + 2) * 8, hipMemcpyDeviceToHost, stream));
    MK_HIP(hipEventRecord(ev1, stream));
    MK_HIP(hipEventSynchronize(ev1));
    const unsigned long long *h = host.as<unsigned long long>();
    total = 0;
    for (uint32_t k = 0; k < kTcSlots; ++k) total += h[k];
    last_slabs = h[kTcSlots];
    last_streamed = h[kTcSlots + 1];
    float t = 0.f;
    MK_HIP(hipEventElapsedTime(&t, ev0, ev1));
    if (ms) *ms = t;
    return MK_OK;
  }

  // hipcub exclusive sum of n + 1 values on the handle's stream, in scan_tmp
  // (of `tmp` bytes at least).
  int exclusive_sum(const unsigned long long *in, unsigned long long *out, size_t tmp) {
    MK_HIP(hipcub::DeviceScan::ExclusiveSum(scan_tmp.ptr, tmp, in, out, int(size_t(g->n) + 1),
                                            stream));
    return MK_OK;
  }
  // (through a word behind finish()'s; a copy and a stream wait cost 8 us more)
  int read_word(const unsigned long long *p, uint64_t &x) {
    constexpr uint32_t at = (kTcSlots + 2) * 2;
    publish_words(reinterpret_cast<const uint32_t *>(p), static_cast<uint32_t *>(host.dev) + at, 2,
                  ++word_seq, stream);
    if (int r = host_wait_word(host.as<uint32_t>() + at + 2, word_seq, stream)) return r;
    x = host.as<volatile uint64_t>()[kTcSlots + 2];
    return MK_OK;
  }
  // The static count's scratch over sorted rows (uplist, scan_tmp and grabs
  // are the plain lists' too).
  uint64_t wedge_scratch() const {
    uint64_t sum = 0;
    for (const DevBuf *b : {&ranks, &rows, &raw, &slot, &units, &uplist, &scan_tmp, &grabs})
      sum += b->bytes;
    return sum;
  }
  // Grow a buffer of it, with an eighth to spare where nothing bounds it;
  // false when memory is short, or past the bound (0: none).
  bool fits(DevBuf &b, uint64_t bytes, uint64_t limit) {
    if (b.ptr && b.bytes >= bytes) return true;
    if (limit) {
      if (wedge_scratch() - b.bytes + std::max<uint64_t>(bytes, 256) > limit) return false;
    } else if (b.ensure(bytes + bytes / 8) == MK_OK) {
      return true;
    }
    if (b.ensure(bytes) == MK_OK) return true;
    (void)hipGetLastError();
    return false;
  }
  void release_wedges() {
    (void)hipStreamSynchronize(stream);
    for (DevBuf *b : {&ranks, &rows, &raw, &slot, &units, &scan_tmp}) b->release();
  }

  // The wedge count queued on the stream (its result in `slots`), or
  // *done = false when device memory for its lists is short (or over the
  // knob "tc_scratch_mb"): nothing is counted then.
  int queue_wedges(bool *done) {
    *done = false;
    const uint32_t n = g->n;
    const uint64_t limit = uint64_t(tune_get("tc_scratch_mb", 0)) << 20;
    if (limit && wedge_scratch() > limit) {  // grown without the bound
      release_wedges();
      uplist.release();
    }
    // ranks: keys and values of the sort by (degree, id), both ways, and
    // the rank of each vertex; rows: places and lengths
    const size_t n1 = size_t(spread_rows(n)) * kSpread + 2;
    if (!fits(ranks, n1 * 16, limit) || !fits(rows, n1 * 32, limit)) return MK_OK;
    uint32_t *rank = ranks.as<uint32_t>(), *ids = rank + n1, *order = ids + n1, *sdeg = order + n1;
    unsigned long long *row0 = rows.as<unsigned long long>(), *off = row0 + n1, *tmp = off + n1;
    uint32_t *len = reinterpret_cast<uint32_t *>(tmp + n1), *ndown = len + n1;
    const unsigned tgrid = blocks_for_threads(n), grid = blocks_for_waves(
        std::min<uint64_t>((uint64_t(n) + 7) / 8, uint64_t(device_cus(g->device)) * 32));
    ProfScope prof(stream, "k_tc_lists", 0.0);
    k_tc_iota<<<tgrid, kBlock, 0, stream>>>(ids, n);
    // degrees are below n (no self-loops, no duplicates)
    int bits = 1;
    while (bits < 32 && (n >> bits)) ++bits;
    size_t need = 0, scan = 0;
    MK_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, need, g->vdeg, sdeg, ids, order, int(n), 0,
                                              bits, stream));
    MK_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, scan, tmp, row0, int(size_t(n) + 1), stream));
    if (!fits(scan_tmp, std::max(need, scan), limit)) return MK_OK;
    MK_HIP(hipcub::DeviceRadixSort::SortPairs(scan_tmp.ptr, need, g->vdeg, sdeg, ids, order,
                                              int(n), 0, bits, stream));
    fill_u64(reinterpret_cast<uint64_t *>(tmp) + n, 0ull, 1, stream);
    k_tc_rank<<<tgrid, kBlock, 0, stream>>>(order, sdeg, n, rank, tmp);
    if (int r = exclusive_sum(tmp, row0, scan)) return r;
    // Up to kSmallTotal stored edges the arrays are made for the most there
    // can be, and the host waits for no length but this one, for none where n
    // alone tells: each wait is some 10 us of a call of 75.
    uint64_t total = uint64_t(n) * (n - 1);
    if (limit || total > kSmallTotal)
      if (int r = read_word(row0 + n, total)) return r;
    const bool small = !limit && total <= kSmallTotal;
    // 4 B a direction here and 4 B below
    if (limit && n1 * 48 + total * 8 > limit) return MK_OK;
    if (!fits(raw, std::max<uint64_t>(total, 1) * (small ? 8 : 4), limit)) return MK_OK;
    fill_u32(len, 0u, 2 * n1, stream);  // and ndown
    const unsigned bgrid = blocks_for_waves(std::min<uint64_t>(
        (uint64_t(g->total_buckets) + 7) / 8, uint64_t(device_cus(g->device)) * 32));
    auto kr = g->weighted ? k_tc_rows<true> : k_tc_rows<false>;
    kr<<<bgrid, kBlock, 0, stream>>>(g->view(), rank, row0, len, raw.as<uint32_t>(),
                                     slots + kTcSlots);
    k_tc_widen<<<blocks_for_threads(uint64_t(n) + 1), kBlock, 0, stream>>>(len, n, false, tmp);
    if (int r = exclusive_sum(tmp, off, scan)) return r;
    uint64_t ups = total;
    if (!small)
      if (int r = read_word(off + n, ups)) return r;
    if (ups == 0) {
      *done = true;
      return MK_OK;
    }
    if (!fits(uplist, ups * 4, limit) || !fits(slot, ups * 4, limit)) return MK_OK;
    k_tc_sort<<<grid, kBlock, 0, stream>>>(row0, len, off, raw.as<uint32_t>(), n,
                                           uplist.as<uint32_t>(), slot.as<uint32_t>(), ndown);
    k_tc_widen<<<blocks_for_threads(uint64_t(n) + 1), kBlock, 0, stream>>>(ndown, n, true, tmp);
    unsigned long long *dof = row0;  // the raw rows' places are done with
    if (int r = exclusive_sum(tmp, dof, scan)) return r;
    uint64_t entries = ups;
    if (!small)
      if (int r = read_word(dof + n, entries)) return r;
    const uint64_t nunits = (entries + kUnit - 1) / kUnit;
    // the lists take the raw rows' memory: two words an entry, at most one
    // entry per undirected edge of a graph that holds both directions
    if (!fits(raw, std::max<uint64_t>(entries, 1) * 8, limit) ||
        !fits(units, std::max<uint64_t>(nunits, 1) * 4, limit) ||
        !fits(grabs, kTakers * 128, limit))
      return MK_OK;
    if (entries) {
      unsigned long long *down = raw.as<unsigned long long>();
      k_tc_down<<<grid, kBlock, 0, stream>>>(len, off, uplist.as<uint32_t>(), slot.as<uint32_t>(),
                                             dof, n, down);
      k_tc_units<<<tgrid, kBlock, 0, stream>>>(dof, n, units.as<uint32_t>());
      uint64_t stride = 1;
      if (nunits > 2) {
        stride = uint64_t(double(nunits) * 0.6180339887) | 1u;
        while (std::gcd(stride, nunits) != 1) stride += 2;
        stride %= nunits;
      }
      fill_u64(grabs.as<uint64_t>(), 0ull, kTakers * 16, stream);
      ProfScope prof2(stream, "k_tc_intersect", 0.0);
      const unsigned wgrid = blocks_for_waves(
          std::min<uint64_t>(nunits, uint64_t(device_cus(g->device)) * 32));
      k_tc_wedges<<<wgrid, kBlock, 0, stream>>>(len, off, uplist.as<uint32_t>(), dof, down,
                                                units.as<uint32_t>(), n, small ? 0 : entries,
                                                nunits, stride,
                                                grabs.as<unsigned long long>(), slots);
    }
    MK_HIP(hipGetLastError());
    *done = true;
    return MK_OK;
  }

  int run_static(float *ms) {
    if (int r = start()) return r;
    bool done = false;
    if (int r = queue_wedges(&done)) return r;
    if (done) {
      uint64_t t = 0;
      if (int r = finish(t, ms)) return r;
      if (profiling_on()) prof_add_bytes("k_tc_lists", 256.0 * double(last_slabs));
      count = t;
      return MK_OK;
    }
    release_wedges();  // the plain lists may need their memory
    return run_static_lists(ms);
  }

  // Static count without the sorted rows: 4 bytes of scratch an undirected
  // edge.
  int run_static_lists(float *ms) {
    fill_u64(reinterpret_cast<uint64_t *>(slots), 0ull, kTcSlots + 2, stream);
    const size_t n = g->n;
    if (int r = kup.ensure((n + 1) * 8)) return r;
    if (int r = koff.ensure((n + 1) * 8)) return r;
    if (int r = grabs.ensure(3 * 8)) return r;
    unsigned long long *K = kup.as<unsigned long long>(), *off = koff.as<unsigned long long>();
    // one vertex counter per pass
    unsigned long long *next = grabs.as<unsigned long long>();
    fill_u64(reinterpret_cast<uint64_t *>(next), 0ull, 3, stream);
    const unsigned grid = blocks_for_waves(
        std::min<uint64_t>((n + kGrab - 1) / kGrab, uint64_t(max_waves) * 2));
    {
      // higher-ranked neighbour lists: count, scan, fill
      ProfScope prof(stream, "k_tc_lists", 0.0);
      fill_u64(reinterpret_cast<uint64_t *>(K) + n, 0ull, 1, stream);
      if (g->weighted)
        k_tc_count_up<true><<<grid, kBlock, 0, stream>>>(g->view(), K, slots + kTcSlots, next);
      else
        k_tc_count_up<false><<<grid, kBlock, 0, stream>>>(g->view(), K, slots + kTcSlots, next);
      size_t tmp = 0;
      MK_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, K, off, int(n + 1), stream));
      if (int r = scan_tmp.ensure(tmp)) return r;
      MK_HIP(hipcub::DeviceScan::ExclusiveSum(scan_tmp.ptr, tmp, K, off, int(n + 1), stream));
      MK_HIP(hipMemcpyAsync(host.ptr, off + n, 8, hipMemcpyDeviceToHost, stream));
      MK_HIP(hipStreamSynchronize(stream));
      const uint64_t total = *host.as<uint64_t>();
      if (int r = uplist.ensure(std::max<uint64_t>(total, 1) * 4)) return r;
      if (g->weighted)
        k_tc_fill_up<true><<<grid, kBlock, 0, stream>>>(g->view(), off, uplist.as<uint32_t>(),
                                                       slots + kTcSlots, next + 1);
      else
        k_tc_fill_up<false><<<grid, kBlock, 0, stream>>>(g->view(), off, uplist.as<uint32_t>(),
                                                        slots + kTcSlots, next + 1);
    }
    {
      ProfScope prof(stream, "k_tc_intersect", 0.0);
      k_tc_intersect<<<grid, kBlock, 0, stream>>>(off, uplist.as<uint32_t>(), g->n, slots,
                                                  slots + kTcSlots + 1, next + 2);
    }
    uint64_t t = 0;
    if (int r = finish(t, ms)) return r;
    if (profiling_on()) {
      // lists: 256 B per slab read (twice), 4 B per neighbour degree, 4 B
      // per list entry written; intersection: 4 B per streamed element and
      // per staged entry, 16 B per vertex (offsets)
      prof_add_bytes("k_tc_lists", 256.0 * double(last_slabs));
      prof_add_bytes("k_tc_intersect", 4.0 * double(last_streamed) + 16.0 * double(n));
    }
    count = t;
    return MK_OK;
  }

  // Changed undirected edges of the batch into the set, their count in m, that
  // of their work items in nitems.
  int collect(const uint32_t *src, const uint32_t *dst, uint32_t n, int op, uint32_t &mask,
              uint32_t &m, uint64_t &nitems) {
    uint32_t cap = 1024;
    while (cap < 2ull * n) cap <<= 1;
    mask = cap - 1;
    if (int r = tab.ensure(size_t(cap) * 8)) return r;
    if (int r = owned.ensure(size_t(std::max(n, 1u)) * 8)) return r;
    fill_u64(tab.as<uint64_t>(), ~0ull, cap, stream);
    fill_u32(n_owned, 0u, 8, stream);
    unsigned long long *n_items = reinterpret_cast<unsigned long long *>(n_owned + 2);
    const bool same = g->last_op == op && g->last_src == src && g->last_dst == dst &&
                      g->status_n == n;
    const uint8_t *st = same ? g->status.as<uint8_t>() : nullptr;
    k_tc_collect<<<blocks_for_threads(n), kBlock, 0, stream>>>(
        g->view(), src, dst, st, n, g->n, tab.as<unsigned long long>(), mask, owned.as<uint2>(),
        n_owned, n_items);
    MK_HIP(hipGetLastError());
    MK_HIP(hipMemcpyAsync(host.ptr, n_owned, 16, hipMemcpyDeviceToHost, stream));
    MK_HIP(hipStreamSynchronize(stream));
    m = host.as<uint32_t>()[0];
    nitems = host.as<uint64_t>()[1];
    if (int r = items.ensure(std::min(nitems, kMaxItems) * 8)) return r;
    if (nitems > kMaxItems)
      if (int r = item_start.ensure(size_t(m) * 8)) return r;
    return MK_OK;
  }

  // Every work item of the m changed edges to `launch` (grid, items, their
  // number), a window after the other.
  template <typename F> void each_window(uint32_t m, uint64_t nitems, const F &launch) {
    unsigned long long *written = reinterpret_cast<unsigned long long *>(n_owned + 4);
    unsigned long long *start =
        nitems > kMaxItems ? item_start.as<unsigned long long>() : nullptr;
    for (uint64_t lo = 0; lo < nitems; lo += kMaxItems) {
      const uint64_t hi = std::min(lo + kMaxItems, nitems);
      k_tc_items<<<blocks_for_threads(m), kBlock, 0, stream>>>(
          g->view(), owned.as<uint2>(), m, items.as<uint2>(), written, start, lo, hi);
      launch(blocks_for_waves(std::min<uint64_t>(hi - lo, uint64_t(max_waves) * 2)),
             items.as<uint2>(), hi - lo);
    }
  }

  int run_incremental(const uint32_t *src, const uint32_t *dst, uint32_t n, float *ms) {
    if (n && (!src || !dst)) return fail(MK_ERR_BAD_ARG, "tc incremental: NULL batch");
    if (int r = start()) return r;
    uint64_t t = 0;
    if (n) {
      uint32_t mask = 0, m = 0;
      uint64_t ni = 0;
      if (int r = collect(src, dst, n, 1, mask, m, ni)) return r;
      if (m) {
        ProfScope prof(stream, "k_tc_inserted", 0.0);
        auto k = g->weighted ? k_tc_inserted<true> : k_tc_inserted<false>;
        each_window(m, ni, [&](unsigned grid, const uint2 *it, uint64_t count) {
          k<<<grid, kBlock, 0, stream>>>(g->view(), owned.as<uint2>(), it, count,
                                         tab.as<unsigned long long>(), mask, slots,
                                         slots + kTcSlots);
        });
      }
    }
    if (int r = finish(t, ms)) return r;
    if (profiling_on()) prof_add_bytes("k_tc_inserted", 256.0 * double(last_slabs));
    count += t / 6;
    return MK_OK;
  }

  int run_decremental(const uint32_t *src, const uint32_t *dst, uint32_t n, float *ms) {
    if (n && (!src || !dst)) return fail(MK_ERR_BAD_ARG, "tc decremental: NULL batch");
    if (int r = start()) return r;
    uint64_t t = 0;
    if (n) {
      uint32_t mask = 0, m = 0;
      uint64_t ni = 0;
      if (int r = collect(src, dst, n, 2, mask, m, ni)) return r;
      if (m) {
        // CSR of the deleted edges (both directions)
        const size_t nv = g->n;
        if (int r = ddeg.ensure((nv + 1) * 4)) return r;
        if (int r = doff.ensure((nv + 1) * 4)) return r;
        if (int r = cursor.ensure(nv * 4)) return r;
        if (int r = dlist.ensure(size_t(m) * 8)) return r;
        fill_u32(ddeg.as<uint32_t>(), 0u, nv + 1, stream);
        fill_u32(cursor.as<uint32_t>(), 0u, nv, stream);
        k_tc_dcount<<<blocks_for_threads(m), kBlock, 0, stream>>>(owned.as<uint2>(), m,
                                                                 ddeg.as<uint32_t>());
        size_t tmp = 0;
        MK_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, ddeg.as<uint32_t>(),
                                                doff.as<uint32_t>(), int(nv + 1), stream));
        if (int r = scan_tmp.ensure(tmp)) return r;
        MK_HIP(hipcub::DeviceScan::ExclusiveSum(scan_tmp.ptr, tmp, ddeg.as<uint32_t>(),
                                                doff.as<uint32_t>(), int(nv + 1), stream));
        k_tc_dfill<<<blocks_for_threads(m), kBlock, 0, stream>>>(
            owned.as<uint2>(), m, doff.as<uint32_t>(), cursor.as<uint32_t>(),
            dlist.as<uint32_t>());
        ProfScope prof(stream, "k_tc_deleted", 0.0);
        auto k = g->weighted ? k_tc_deleted<true> : k_tc_deleted<false>;
        each_window(m, ni, [&](unsigned grid, const uint2 *it, uint64_t count) {
          k<<<grid, kBlock, 0, stream>>>(g->view(), owned.as<uint2>(), it, count,
                                         tab.as<unsigned long long>(), mask,
                                         doff.as<uint32_t>(), dlist.as<uint32_t>(), slots,
                                         slots + kTcSlots);
        });
      }
    }
    if (int r = finish(t, ms)) return r;
    if (profiling_on()) prof_add_bytes("k_tc_deleted", 256.0 * double(last_slabs));
    count -= t / 6;
    return MK_OK;
  }
};

}  // namespace mk

struct mk_tc {
  mk::TC t;
};

using namespace mk;

extern "C" {

int mk_tc_create(mk_graph *g, mk_tc **out) {
  if (!out) return fail(MK_ERR_BAD_ARG, "mk_tc_create: out is NULL");
  *out = nullptr;
  if (!g) return fail(MK_ERR_BAD_ARG, "mk_tc_create: NULL graph");
  mk_tc *h = new mk_tc();
  int r = h->t.init(g);
  if (r) {
    h->t.destroy();
    delete h;
    return r;
  }
  g->users++;
  *out = h;
  return MK_OK;
}

int mk_tc_destroy(mk_tc *t) {
  if (!t) return fail(MK_ERR_BAD_ARG, "mk_tc_destroy: NULL handle");
  t->t.g->users--;
  t->t.destroy();
  delete t;
  return MK_OK;
}

int mk_tc_static(mk_tc *t, float *ms) {
  if (!t) return fail(MK_ERR_BAD_ARG, "mk_tc_static: NULL handle");
  if (int r = graph_settle(t->t.g)) return r;
  return t->t.run_static(ms);
}

int mk_tc_incremental(mk_tc *t, const uint32_t *src, const uint32_t *dst, uint32_t n,
                      float *ms) {
  if (!t) return fail(MK_ERR_BAD_ARG, "mk_tc_incremental: NULL handle");
  if (int r = graph_settle(t->t.g)) return r;
  if (int r = graph_failed_batch(t->t.g, src, dst, n)) return r;
  return t->t.run_incremental(src, dst, n, ms);
}

int mk_tc_decremental(mk_tc *t, const uint32_t *src, const uint32_t *dst, uint32_t n,
                      float *ms) {
  if (!t) return fail(MK_ERR_BAD_ARG, "mk_tc_decremental: NULL handle");
  if (int r = graph_settle(t->t.g)) return r;
  if (int r = graph_failed_batch(t->t.g, src, dst, n)) return r;
  return t->t.run_decremental(src, dst, n, ms);
}

int mk_tc_count(mk_tc *t, uint64_t *count) {
  if (!t || !count) return fail(MK_ERR_BAD_ARG, "mk_tc_count: NULL argument");
  *count = t->t.count;
  return MK_OK;
}

}  // extern "C"
