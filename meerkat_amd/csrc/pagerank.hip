// PageRank (FP32 ranks, FP64 reductions) over a slab-hash in-adjacency.
//
// Reference: include/Algorithms/PageRank.cuh:9-68 and impl/PageRankImpl.cuh:
//   contrib[v] = outdeg[v] ? PR[v] / outdeg[v] : 0           (:133-144)
//   acc        = sum_{outdeg(x) = 0} PR[x] / N                 (:89-107)
//   PR'[u]     = (1 - d) / N + d * sum_{v in in(u)} contrib[v] + d * acc
//                                                    (:3-62, :109-115, :193)
//   delta      = sum |PR' - PR|; loop while delta > margin && it < max_iter
//                                                    (:117-131, :173)
// Ranks start at 1/N (PageRank.cuh:42-43); Static, Incremental and
// Decremental all continue from the current ranks (warm start), after the
// out-degree fix-up for the batch (CheckPresent, :64-87).
//
// Method: one fused kernel per iteration computes PR', the next
// contributions, the next dangling mass and the L1 delta (FP64 partial sums
// spread over kSlots addresses).  Each iteration kernel first evaluates the
// stopping rule from the previous kernel's delta, so the host launches
// iterations in groups without waiting and the iteration count is exactly
// the reference's.  Vertices whose in-adjacency spans more than kHubBuckets
// buckets have their buckets spread over all waves (partial sums added to a
// per-hub FP64 accumulator) and are finished by a second, small kernel.
//
// In-adjacency: either a graph holding reversed edges, as the reference's
// RevUnweightedEdgePolicyT graph (PageRank.cuh:11; the driver inserts (dst,
// src), src/PageRank.cu:137), whose out-degrees are host-provided and fixed
// up per batch; or a graph created with MK_GRAPH_REVERSE, whose mirror is
// the in-adjacency and whose live out-degree array is exact.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <vector>

#include "profile.hpp"
#include "readback.hpp"
#include "slabhash.hpp"

namespace mk {

constexpr uint32_t kSlots = 64;       // FP64 partial-sum addresses
constexpr uint32_t kHubBuckets = 4;   // more in-buckets than this: hub path
constexpr uint32_t kPrBatch = 4;      // slab loads in flight per wave

// Packed edge list of a call (PrPlan): destinations in bins of up to
// 2^kBinMaxBits vertices, sources in parts of 2^19 (2^20) vertices.
constexpr uint32_t kBinMaxBits = 12;
constexpr uint32_t kMaxParts = 64;
constexpr uint32_t kChunkBuckets = 64;  // in-buckets per chunk of a bin
constexpr uint32_t kPlanBlock = 1024;   // threads of k_pr_iterate_bins

struct PrState {
  double delta[3][kSlots];   // L1 delta of iteration i in [i % 3]
  double dang[3][kSlots];    // dangling mass of the ranks iteration i reads
  uint32_t iters;            // iterations completed in this call
  uint32_t stopped;          // stopping rule met
  double last_delta;
};

struct PrView {
  float *pr[2];
  float *contrib[2];
  const uint32_t *outdeg;
  PrState *st;
  const uint32_t *hub_vertex;  // hub index -> vertex
  const uint32_t *hub_start;   // hub index -> first work item (sorted)
  double *hub_acc;             // per hub in-sum of the running iteration
  uint32_t n_hubs, hub_items;
  uint32_t n;
  float damping;
  double margin;
  uint32_t max_iter;
};

// The in-adjacency packed for the iterations of one call.  Edge (v -> u) is
// one word: u's place in its bin (bin_bits) above v's place in its part
// (part_bits; together at most 32).  Words are ordered by (bin, part); the
// bin's chunks of kChunkBuckets buckets share out each cell, so `cell` (the
// exclusive sum of the per-(bin, part, chunk) counts) places every chunk's
// words and holds the cell bounds.
struct PrPlan {
  const uint32_t *bin_chunk0;      // bins + 1: a bin's first chunk
  unsigned long long *count;       // chunks * parts + 1 (the last 0)
  unsigned long long *cell;        // their exclusive sum
  uint32_t *words;
  uint2 *items;                    // work items of k_pr_iterate_bins: (bin, sub-range)
  uint32_t *bin_items;             // items of each bin
  uint32_t *n_items;
  double *acc;                     // n: sums of the bins split into items (zero between uses)
  uint32_t *arrived;               // per bin: items done (zero between uses)
  uint32_t bins, bin_bits, parts, part_bits, chunks;
};

MK_DEV unsigned long long cell_start(const PrPlan &L, uint32_t bin, uint32_t part) {
  const uint32_t c0 = L.bin_chunk0[bin], c1 = L.bin_chunk0[bin + 1];
  return L.cell[size_t(c0) * L.parts + size_t(part) * (c1 - c0)];
}

MK_DEV unsigned long long bin_end(const PrPlan &L, uint32_t bin) {
  return bin + 1 < L.bins ? cell_start(L, bin + 1, 0) : L.cell[size_t(L.chunks) * L.parts];
}

MK_DEV double wave_sum_slots(const double *slots) {
  double x = slots[lane_id()];
  return wave_sum_f64(x);
}

MK_DEV void add_slot(double *slots, double v) {
  if (v != 0.0) atomicAdd(&slots[blockIdx.x % kSlots], v);
}

// Stopping rule at the start of iteration i; every thread evaluates it.
MK_DEV bool pr_should_stop(const PrView &P, uint32_t i) {
  if (P.st->stopped) return true;
  if (i >= P.max_iter) return true;
  if (i == 0) return false;  // the reference's loop starts with delta = 1
  const double d = wave_sum_slots(P.st->delta[(i - 1) % 3]);
  return !(d > P.margin);
}

// Sum of contrib over one in-chain (first slab word x loaded).
template <bool MAP>
MK_DEV float chain_sum(const GraphView &R, const float *contrib, uint32_t x, uint32_t &slabs) {
  const uint32_t lane = lane_id();
  const bool key_lane = (key_mask<MAP>() >> lane) & 1ull;
  float acc = 0.f;
  for (;;) {
    ++slabs;
    if (key_lane && x < kTomb) acc += contrib[x];
    const uint32_t nx = read_lane(x, kNextLane);
    if (nx == kEmpty) break;
    x = slab_ptr(R.pool, nx)[lane];
  }
  return wave_sum_f32(acc);
}

// Clears every reduction slot and the iteration counters of a compute call
// (one block of kSlots threads, launched before k_pr_prepare adds into
// dang[0]).
__global__ void k_pr_reset(PrState *st) {
  const uint32_t t = threadIdx.x;
  for (uint32_t k = 0; k < 3; ++k) {
    st->delta[k][t] = 0.0;
    st->dang[k][t] = 0.0;
  }
  if (t == 0) {
    st->iters = 0;
    st->stopped = 0;
  }
}

// Initial contributions and dangling mass of the current ranks.
__global__ void __launch_bounds__(kBlock) k_pr_prepare(PrView P, uint32_t cur) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  double dang = 0.0;
  if (i < P.n) {
    const float r = P.pr[cur][i];
    const uint32_t od = P.outdeg[i];
    P.contrib[cur][i] = od ? r / float(od) : 0.f;
    if (od == 0) dang = double(r);
  }
  dang = wave_sum_f64(dang);
  if (lane_id() == 0) add_slot(P.st->dang[0], dang);
}

// One PageRank iteration i over non-hub vertices, plus the hubs' partial
// in-sums.  Reads pr/contrib[(cur + i) & 1], writes the other buffers.
template <bool MAP>
__global__ void __launch_bounds__(kBlock)
    k_pr_iterate(GraphView R, PrView P, uint32_t cur, uint32_t i) {
  if (pr_should_stop(P, i)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) P.st->stopped = 1;
    return;
  }
  const uint32_t lane = lane_id();
  const uint32_t gw = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t W = (gridDim.x * blockDim.x) >> 6;
  const uint32_t a = (cur + i) & 1u, b = a ^ 1u;
  if (blockIdx.x == 0 && threadIdx.x < kSlots) {
    P.st->delta[(i + 1) % 3][threadIdx.x] = 0.0;  // written by iteration i + 1
    P.st->dang[(i + 2) % 3][threadIdx.x] = 0.0;   // written by iteration i + 1
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) P.st->iters = i + 1;
  const float *contrib = P.contrib[a];
  const float base = (1.0f - P.damping) / float(P.n);
  const float dang = float(wave_sum_slots(P.st->dang[i % 3]) / double(P.n));
  uint32_t slabs = 0;
  // hub buckets: work items spread over all waves, partial sums per hub
  for (uint32_t t0 = gw * 64; t0 < P.hub_items; t0 += W * 64) {
    const uint32_t t = t0 + lane;
    bool act = t < P.hub_items;
    uint32_t h = 0, bk = 0;
    if (act) {
      uint32_t lo = 0, hi = P.n_hubs;
      while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (P.hub_start[mid] <= t) lo = mid;
        else hi = mid;
      }
      h = lo;
      bk = R.bucket_off[P.hub_vertex[h]] + (t - P.hub_start[h]);
    }
    uint64_t m = ballot(act);
    while (m) {
      uint32_t js[kPrBatch];
      uint32_t c = 0;
#pragma unroll
      for (uint32_t k = 0; k < kPrBatch; ++k) {
        js[k] = m ? ffs64(m) : 0u;
        if (m) {
          m &= m - 1;
          c = k + 1;
        }
      }
      uint32_t x[kPrBatch];
#pragma unroll
      for (uint32_t k = 0; k < kPrBatch; ++k)
        x[k] = k < c ? R.heads[size_t(read_lane(bk, js[k])) * kSlabWords + lane] : kEmpty;
#pragma unroll
      for (uint32_t k = 0; k < kPrBatch; ++k) {
        if (k >= c) continue;
        const float s = chain_sum<MAP>(R, contrib, x[k], slabs);
        const uint32_t hk = read_lane(h, js[k]);  // with every lane active
        if (lane == 0) atomicAdd(&P.hub_acc[hk], double(s));
      }
    }
  }
  // ordinary vertices: 64 per wave step, one lane per vertex
  double delta = 0.0, dnext = 0.0;
  for (uint32_t u0 = gw * 64; u0 < P.n; u0 += W * 64) {
    const uint32_t u = u0 + lane;
    bool act = u < P.n;
    uint32_t b0 = 0, nb = 0;
    if (act) {
      b0 = R.bucket_off[u];
      nb = R.bucket_off[u + 1] - b0;
      if (nb > kHubBuckets) act = false;  // finished by k_pr_hubs
    }
    float acc = 0.f;
    for (uint32_t k = 0; ballot(act && nb > k); ++k) {
      uint64_t m = ballot(act && nb > k);
      while (m) {
        uint32_t js[kPrBatch];
        uint32_t c = 0;
#pragma unroll
        for (uint32_t q = 0; q < kPrBatch; ++q) {
          js[q] = m ? ffs64(m) : 0u;
          if (m) {
            m &= m - 1;
            c = q + 1;
          }
        }
        uint32_t x[kPrBatch];
#pragma unroll
        for (uint32_t q = 0; q < kPrBatch; ++q)
          x[q] = q < c ? R.heads[size_t(read_lane(b0, js[q]) + k) * kSlabWords + lane] : kEmpty;
#pragma unroll
        for (uint32_t q = 0; q < kPrBatch; ++q) {
          if (q >= c) continue;
          const float s = chain_sum<MAP>(R, contrib, x[q], slabs);
          if (lane == js[q]) acc += s;
        }
      }
    }
    if (act) {
      const float x = base + P.damping * acc + P.damping * dang;
      const float old = P.pr[a][u];
      delta += double(fabsf(x - old));
      P.pr[b][u] = x;
      const uint32_t od = P.outdeg[u];
      P.contrib[b][u] = od ? x / float(od) : 0.f;
      if (od == 0) dnext += double(x);
    }
  }
  delta = wave_sum_f64(delta);
  dnext = wave_sum_f64(dnext);
  if (lane == 0) {
    add_slot(P.st->delta[i % 3], delta);
    add_slot(P.st->dang[(i + 1) % 3], dnext);
  }
}

// Finish the hub vertices of iteration i (after k_pr_iterate).
__global__ void __launch_bounds__(kBlock) k_pr_hubs(PrView P, uint32_t cur, uint32_t i) {
  // k_pr_iterate of this iteration already evaluated the rule and set
  // `stopped`; iters tells whether iteration i ran
  if (P.st->iters != i + 1 || P.st->stopped) return;
  const uint32_t a = (cur + i) & 1u, b = a ^ 1u;
  const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
  const float base = (1.0f - P.damping) / float(P.n);
  const float dang = float(wave_sum_slots(P.st->dang[i % 3]) / double(P.n));
  double delta = 0.0, dnext = 0.0;
  if (h < P.n_hubs) {
    const uint32_t u = P.hub_vertex[h];
    const float x = base + P.damping * float(P.hub_acc[h]) + P.damping * dang;
    P.hub_acc[h] = 0.0;
    delta = double(fabsf(x - P.pr[a][u]));
    P.pr[b][u] = x;
    const uint32_t od = P.outdeg[u];
    P.contrib[b][u] = od ? x / float(od) : 0.f;
    if (od == 0) dnext = double(x);
  }
  delta = wave_sum_f64(delta);
  dnext = wave_sum_f64(dnext);
  if (lane_id() == 0) {
    add_slot(P.st->delta[i % 3], delta);
    add_slot(P.st->dang[(i + 1) % 3], dnext);
  }
}

// Has the call ended with iteration i - 1?  (One wave.)
__global__ void __launch_bounds__(64) k_pr_ended(PrView P, uint32_t i) {
  if (pr_should_stop(P, i) && threadIdx.x == 0) P.st->stopped = 1;
}

// Chunk `c`'s bin (the last with bin_chunk0 <= c).
MK_DEV uint32_t chunk_bin(const PrPlan &L, uint32_t c) {
  uint32_t lo = 0, hi = L.bins;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (L.bin_chunk0[mid] <= c) lo = mid;
    else hi = mid;
  }
  return lo;
}

// One pass over the slabs of the in-adjacency, a wave per chunk and an
// 8-lane group per bucket (eight slabs in flight per wave; a slab's keys
// sit two to a lane in load_words' layout, so most key rounds have 32 lanes
// at work where a wave per slab has as many as the slab has keys).
// FILL = false counts the keys of every (bin, part, chunk); FILL = true
// writes the packed words at the scanned places.  Bound by the 256 bytes
// read per bucket: ER 4.2M x 33.5M (1.07 GB of slabs) takes 0.20 ms to
// count (5.3 TB/s) and, writing 134 MB in short runs, 0.46 ms to fill.
template <bool MAP, bool FILL>
__global__ void __launch_bounds__(kBlock) k_pr_pack(GraphView R, PrPlan L) {
  __shared__ uint32_t cnt[kBlock / 64][kMaxParts];
  __shared__ unsigned long long base[kBlock / 64][kMaxParts];
  const uint32_t lane = lane_id(), gl = group_lane(), w = threadIdx.x >> 6;
  const uint32_t gw = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t W = (gridDim.x * blockDim.x) >> 6;
  for (uint32_t c = gw; c < L.chunks; c += W) {
    const uint32_t bin = chunk_bin(L, c);
    const uint32_t c0 = L.bin_chunk0[bin], nc = L.bin_chunk0[bin + 1] - c0;
    const size_t cell0 = size_t(c0) * L.parts + (c - c0);
    if (lane < L.parts) {
      cnt[w][lane] = 0u;
      if (FILL) base[w][lane] = L.cell[cell0 + size_t(lane) * nc];
    }
    __builtin_amdgcn_wave_barrier();
    const uint32_t v0 = bin << L.bin_bits;
    const uint32_t v1 = bin + 1 < L.bins ? v0 + (1u << L.bin_bits) : R.n;
    const uint32_t b0 = R.bucket_off[v0] + (c - c0) * kChunkBuckets;
    const uint32_t b1 = min(b0 + kChunkBuckets, R.bucket_off[v1]);
    for (uint32_t b = b0 + lane / kGroupLanes; b < b1; b += kGroupsPerWave) {
      const uint32_t hi = FILL ? (R.bucket_owner[b] - v0) << L.part_bits : 0u;
      const uint32_t *slab = R.heads + size_t(b) * kSlabWords;
      for (;;) {
        uint32_t x[kWordsPerLane];
        load_words(slab + kWordsPerLane * gl, x);
#pragma unroll
        for (uint32_t k = 0; k < kWordsPerLane; ++k) {
          if (!key_word<MAP>(kWordsPerLane * gl + k) || x[k] >= kTomb) continue;
          const uint32_t part = x[k] >> L.part_bits;
          const uint32_t at = atomicAdd(&cnt[w][part], 1u);
          if (FILL)
            L.words[base[w][part] + at] = hi | (x[k] & ((1u << L.part_bits) - 1u));
        }
        const uint32_t nx = group_read(x[kWordsPerLane - 1], kGroupLanes - 1);
        if (nx == kEmpty) break;
        slab = slab_ptr(R.pool, nx);
      }
    }
    __builtin_amdgcn_wave_barrier();
    if (!FILL && lane < L.parts) L.count[cell0 + size_t(lane) * nc] = cnt[w][lane];
    __builtin_amdgcn_wave_barrier();
  }
}

// Work items: a bin of more than `cap` words is cut into equal sub-ranges
// of at most `cap` (RMAT's first bin of 4096 vertices holds 6% of the
// edges).  One block.
__global__ void __launch_bounds__(kPlanBlock) k_pr_items(PrPlan L, uint32_t cap) {
  __shared__ uint32_t next;
  if (threadIdx.x == 0) next = 0;
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < L.bins; b += blockDim.x) {
    const unsigned long long cnt = bin_end(L, b) - cell_start(L, b, 0);
    const uint32_t k = cnt ? uint32_t((cnt + cap - 1) / cap) : 1u;
    const uint32_t at = atomicAdd(&next, k);
    L.bin_items[b] = k;
    for (uint32_t i = 0; i < k; ++i) L.items[at + i] = make_uint2(b, i);
  }
  __syncthreads();
  if (threadIdx.x == 0) *L.n_items = next;
}

// Iteration i over the packed words, a block per work item: each word's
// source contribution is added to its destination's FP64 sum in LDS, part
// after part, so that blocks running together gather from neighbouring
// parts (an XCD's L2 holds 4 MB), then the block finishes its bin's
// vertices.  Items of a split bin add their sums to L.acc and the last of
// them to arrive finishes the bin.  Against the walk over the slabs
// (k_pr_iterate) this reads 4 bytes an edge instead of 256 a bucket, and
// gathers from L2 instead of the memory side; it is bound by the L2's
// request rate (a request per word).  MI355X, an iteration: ER 4.2M x 33.5M
// 510 -> 203 us, RMAT 4.2M x 33M 207 us, RMAT 500k x 3.9M 33 us.
__global__ void __launch_bounds__(kPlanBlock)
    k_pr_iterate_bins(PrView P, PrPlan L, uint32_t cur, uint32_t i) {
  if (pr_should_stop(P, i)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) P.st->stopped = 1;
    return;
  }
  __shared__ double acc[1u << kBinMaxBits];
  __shared__ uint32_t bound[kMaxParts + 1];
  __shared__ uint32_t last;
  const uint32_t t = threadIdx.x;
  const uint32_t a = (cur + i) & 1u, b = a ^ 1u;
  if (blockIdx.x == 0 && t < kSlots) {
    P.st->delta[(i + 1) % 3][t] = 0.0;  // written by iteration i + 1
    P.st->dang[(i + 2) % 3][t] = 0.0;   // written by iteration i + 1
  }
  if (blockIdx.x == 0 && t == 0) P.st->iters = i + 1;
  if (blockIdx.x >= *L.n_items) return;
  const uint2 it = L.items[blockIdx.x];
  const uint32_t bin = it.x, parts_of = L.bin_items[bin];
  const uint32_t bsize = 1u << L.bin_bits, v0 = bin << L.bin_bits;
  for (uint32_t k = t; k < bsize; k += kPlanBlock) acc[k] = 0.0;
  // the bin's cell bounds, relative to its first word
  const unsigned long long s0 = cell_start(L, bin, 0);
  for (uint32_t p = t; p <= L.parts; p += kPlanBlock)
    bound[p] = uint32_t((p < L.parts ? cell_start(L, bin, p) : bin_end(L, bin)) - s0);
  __syncthreads();
  const uint32_t total = bound[L.parts], each = (total + parts_of - 1) / parts_of;
  const uint32_t r0 = min(each * it.y, total), r1 = min(r0 + each, total);
  // each thread takes four consecutive words at a time, from the 16-byte
  // boundary below the first; the next four are in flight meanwhile
  const uint32_t skip = uint32_t((s0 + r0) & 3ull);
  const uint4 *wp = reinterpret_cast<const uint4 *>(L.words + (s0 + r0 - skip));
  const uint32_t end = r1 - r0 + skip;  // words of this item, skipped ones included
  const uint32_t mask = (1u << L.part_bits) - 1u;
  const float *contrib = P.contrib[a];
  uint32_t part = 0;
  uint4 nxt = t * 4 < end ? wp[t] : make_uint4(0u, 0u, 0u, 0u);
  for (uint32_t k = t * 4; k < (end + 255) / 256 * 256; k += kPlanBlock * 4) {
    const uint32_t x[4] = {nxt.x, nxt.y, nxt.z, nxt.w};
    const uint32_t kn = k + kPlanBlock * 4;
    if (kn < end) nxt = wp[kn / 4];
    float v[4];
    bool in[4];
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      in[q] = k + q >= skip && k + q < end;
      v[q] = 0.f;
      if (in[q]) {
        const uint32_t at = r0 + k + q - skip;
        while (at >= bound[part + 1]) ++part;
        v[q] = contrib[(part << L.part_bits) | (x[q] & mask)];
      }
    }
    // words of one destination follow each other (a vertex's slabs are
    // packed one after another): equal neighbours are added here, and a
    // wave that holds one destination only (a hub's words) adds its sum
    // once; one FP64 add per word on a hub's sum would serialise
    double s = 0.0;
    uint32_t d = kEmpty;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
      if (!in[q]) continue;
      const uint32_t dq = x[q] >> L.part_bits;
      if (dq != d) {
        if (d != kEmpty) unsafeAtomicAdd(&acc[d], s);
        d = dq;
        s = 0.0;
      }
      s += double(v[q]);
    }
    const uint32_t d0 = first_lane_val(d);
    if (ballot(d == d0) == ~0ull) {
      s = wave_sum_f64(s);
      if (lane_id() == 0 && d0 != kEmpty) unsafeAtomicAdd(&acc[d0], s);
    } else if (d != kEmpty) {
      unsafeAtomicAdd(&acc[d], s);
    }
  }
  __syncthreads();
  if (parts_of > 1) {
    for (uint32_t k = t; k < bsize; k += kPlanBlock)
      if (acc[k] != 0.0) unsafeAtomicAdd(&L.acc[v0 + k], acc[k]);
    // the sums are added, read and cleared by device-scope accesses only, so
    // waiting for one's own is enough; a fence would write back the L2
    // (RMAT 4.2M x 33M, ~680 split items: 0.43 ms of an iteration)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (t == 0) last = atomicAdd(&L.arrived[bin], 1u) + 1u == parts_of ? 1u : 0u;
    __syncthreads();
    if (!last) return;
    if (t == 0) coherent_store(&L.arrived[bin], 0u);
    for (uint32_t k = t; k < bsize && v0 + k < P.n; k += kPlanBlock) {
      acc[k] = __hip_atomic_load(&L.acc[v0 + k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(&L.acc[v0 + k], 0.0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    // each thread finishes the vertices that it read: no barrier
  }
  const float base = (1.0f - P.damping) / float(P.n);
  const float dang = float(wave_sum_slots(P.st->dang[i % 3]) / double(P.n));
  double delta = 0.0, dnext = 0.0;
  for (uint32_t k = t; k < bsize && v0 + k < P.n; k += kPlanBlock) {
    const uint32_t u = v0 + k;
    const float x = base + P.damping * float(acc[k]) + P.damping * dang;
    delta += double(fabsf(x - P.pr[a][u]));
    P.pr[b][u] = x;
    const uint32_t od = P.outdeg[u];
    P.contrib[b][u] = od ? x / float(od) : 0.f;
    if (od == 0) dnext += double(x);
  }
  delta = wave_sum_f64(delta);
  dnext = wave_sum_f64(dnext);
  // one add per block and sum, through the waves' slots of `acc`
  __syncthreads();
  if (lane_id() == 0) {
    acc[(t >> 6) * 2] = delta;
    acc[(t >> 6) * 2 + 1] = dnext;
  }
  __syncthreads();
  if (t < 64) {
    constexpr uint32_t nw = kPlanBlock / 64;
    delta = wave_sum_f64(t < nw ? acc[t * 2] : 0.0);
    dnext = wave_sum_f64(t < nw ? acc[t * 2 + 1] : 0.0);
    if (t == 0) {
      add_slot(P.st->delta[i % 3], delta);
      add_slot(P.st->dang[(i + 1) % 3], dnext);
    }
  }
}

// Out-degree fix-up for a batch: +-1 for each edge the last mutation applied.
__global__ void k_pr_fix_outdeg(uint32_t *outdeg, const uint32_t *src, const uint8_t *status,
                                uint32_t n, int delta) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && status[i] == MK_EDGE_APPLIED) atomicAdd(outdeg + src[i], uint32_t(delta));
}

// Out-degree recount from the in-adjacency: every live key v of an
// in-bucket is one out-edge of v.
template <bool MAP>
__global__ void __launch_bounds__(kBlock) k_pr_recount(GraphView R, uint32_t *outdeg) {
  const uint32_t lane = lane_id();
  const uint32_t gw = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t W = (gridDim.x * blockDim.x) >> 6;
  const bool key_lane = (key_mask<MAP>() >> lane) & 1ull;
  for (uint32_t bk = gw; bk < R.total_buckets; bk += W) {
    uint32_t x = R.heads[size_t(bk) * kSlabWords + lane];
    for (;;) {
      if (key_lane && x < kTomb) atomicAdd(outdeg + x, 1u);
      const uint32_t nx = read_lane(x, kNextLane);
      if (nx == kEmpty) break;
      x = slab_ptr(R.pool, nx)[lane];
    }
  }
}

__global__ void k_fill_f32(float *p, float v, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

struct PageRank {
  mk_graph *g = nullptr;   // graph passed at create
  mk_graph *in = nullptr;  // in-adjacency (g, or g's mirror)
  bool exact_outdeg = false;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  float *pr[2] = {nullptr, nullptr};
  float *contrib[2] = {nullptr, nullptr};
  uint32_t *outdeg = nullptr;
  PrState *st = nullptr;
  uint32_t *hub_vertex = nullptr, *hub_start = nullptr;
  double *hub_acc = nullptr;
  uint32_t n_hubs = 0, hub_items = 0;
  uint32_t cur = 0;
  float damping = 0.85f;
  float margin = 1e-7f;
  uint32_t max_iter = 100;
  HostBuf host;
  uint32_t last_iters = 0;
  double last_delta = 0.0;
  int max_waves = 0;
  // packed in-adjacency of the running call (build_plan): buffers kept with
  // the handle, contents rebuilt by every call that uses them
  PrPlan plan{};
  DevBuf plan_chunk0, plan_cell, plan_scan, plan_words, plan_items, plan_acc;

  PrView view() const {
    PrView v;
    v.pr[0] = pr[0];
    v.pr[1] = pr[1];
    v.contrib[0] = contrib[0];
    v.contrib[1] = contrib[1];
    v.outdeg = outdeg;
    v.st = st;
    v.hub_vertex = hub_vertex;
    v.hub_start = hub_start;
    v.hub_acc = hub_acc;
    v.n_hubs = n_hubs;
    v.hub_items = hub_items;
    v.n = g->n;
    v.damping = damping;
    v.margin = double(margin);
    v.max_iter = max_iter;
    return v;
  }

  int init(mk_graph *graph, float d, float eps, uint32_t iters, const uint32_t *host_outdeg) {
    g = graph;
    in = g->rev ? g->rev : g;
    exact_outdeg = g->rev != nullptr;
    damping = d;
    margin = eps;
    max_iter = iters;
    const size_t n = g->n;
    MK_HIP(hipSetDevice(g->device));
    MK_HIP(hipStreamCreate(&stream));
    loop_stream_add(g->device, stream, 1);
    MK_HIP(hipEventCreate(&ev0));
    MK_HIP(hipEventCreate(&ev1));
    for (int k = 0; k < 2; ++k) {
      MK_HIP(hipMalloc(&pr[k], n * 4));
      MK_HIP(hipMalloc(&contrib[k], n * 4));
    }
    MK_HIP(hipMalloc(&outdeg, n * 4));
    MK_HIP(hipMalloc(&st, sizeof(PrState)));
    if (int r = host.ensure(sizeof(PrState))) return r;
    // hubs: vertices with more than kHubBuckets in-buckets (bucket counts are
    // fixed at graph creation)
    std::vector<uint32_t> hv, hs;
    uint64_t items = 0;
    const std::vector<uint32_t> &off = in->bucket_off_host;
    for (uint32_t v = 0; v < g->n; ++v) {
      const uint32_t nb = off[v + 1] - off[v];
      if (nb > kHubBuckets) {
        hv.push_back(v);
        hs.push_back(uint32_t(items));
        items += nb;
      }
    }
    n_hubs = uint32_t(hv.size());
    hub_items = uint32_t(items);
    MK_HIP(hipMalloc(&hub_vertex, std::max<size_t>(hv.size(), 1) * 4));
    MK_HIP(hipMalloc(&hub_start, std::max<size_t>(hs.size(), 1) * 4));
    MK_HIP(hipMalloc(&hub_acc, std::max<size_t>(hv.size(), 1) * 8));
    if (n_hubs) {
      MK_HIP(hipMemcpy(hub_vertex, hv.data(), hv.size() * 4, hipMemcpyHostToDevice));
      MK_HIP(hipMemcpy(hub_start, hs.data(), hs.size() * 4, hipMemcpyHostToDevice));
    }
    fill_u64(reinterpret_cast<uint64_t *>(hub_acc), 0ull, std::max<uint32_t>(n_hubs, 1), stream);
    k_fill_f32<<<blocks_for_threads(n), kBlock, 0, stream>>>(pr[0], 1.0f / float(n), g->n);
    if (exact_outdeg) {
      MK_HIP(hipMemcpyAsync(outdeg, g->vdeg, n * 4, hipMemcpyDeviceToDevice, stream));
    } else if (host_outdeg) {
      MK_HIP(hipMemcpyAsync(outdeg, host_outdeg, n * 4, hipMemcpyHostToDevice, stream));
    } else {
      if (int r = recount()) return r;
    }
    MK_HIP(hipStreamSynchronize(stream));
    // the iteration gathers 4-byte contributions at random: as many waves
    // as a CU holds (`pr_waves_per_cu`, 32) keep the most loads in flight
    const void *kern = in->weighted ? reinterpret_cast<const void *>(&k_pr_iterate<true>)
                                    : reinterpret_cast<const void *>(&k_pr_iterate<false>);
    MK_HIP(resident_waves(g->device, kern, int(tune_get("pr_waves_per_cu", 32)), &max_waves));
    cur = 0;
    return MK_OK;
  }

  int recount() {
    fill_u32(outdeg, 0u, g->n, stream);
    const unsigned grid = blocks_for_waves(std::min<uint64_t>(in->total_buckets,
                                                              uint64_t(device_cus(g->device)) * 16));
    if (in->weighted)
      k_pr_recount<true><<<grid, kBlock, 0, stream>>>(in->view(), outdeg);
    else
      k_pr_recount<false><<<grid, kBlock, 0, stream>>>(in->view(), outdeg);
    MK_HIP(hipGetLastError());
    return MK_OK;
  }

  void destroy() {
    (void)hipSetDevice(g->device);
    if (stream) (void)hipStreamSynchronize(stream);
    for (int k = 0; k < 2; ++k) {
      (void)hipFree(pr[k]);
      (void)hipFree(contrib[k]);
    }
    (void)hipFree(outdeg);
    (void)hipFree(st);
    (void)hipFree(hub_vertex);
    (void)hipFree(hub_start);
    (void)hipFree(hub_acc);
    for (DevBuf *b : {&plan_chunk0, &plan_cell, &plan_scan, &plan_words, &plan_items, &plan_acc})
      b->release();
    host.release();
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) {
      loop_stream_add(g->device, stream, -1);
      (void)hipStreamDestroy(stream);
    }
  }

  // The packed word has to have room for its two indexes.
  bool plan_fits() const { return g->n <= (kMaxParts << 20); }

  // Pack the in-adjacency as it is now.  Returns false, with nothing left
  // in error, when device memory for it is short: the caller goes on over
  // the slabs.
  bool build_plan(unsigned &grid) {
    const GraphView R = in->view();
    if (!plan.bins) {
      // Bins of up to 2^12 vertices, at least 256 of them: 200k / 500k / 1M /
      // 4.2M vertices ran fastest (ER and RMAT) at 2^9..2^10 / 2^10 / 2^11 /
      // 2^12 a bin, 1.1 to 2 times slower two steps away.
      uint32_t bits = 8;
      while (bits < kBinMaxBits && (g->n >> (bits + 1)) >= 256) ++bits;
      // Fewer vertices with many edges each: smaller bins, so that the
      // device is full (some 20 keys a bucket of a map, 40 of a set).  A
      // clique of 2000, 64 of 300: calls of several iterations 1.05 and 0.61
      // ms with 8 and 75 bins, 0.50 and 0.56 with 63 and 300 (walks over the
      // slabs 0.46 and 0.56).
      const uint64_t keys = uint64_t(in->total_buckets) * (in->weighted ? 20 : 40);
      while (bits > 5 && (g->n >> bits) < 256 && (keys >> 14) > (g->n >> bits)) --bits;
      PrPlan L{};
      L.bin_bits = bits;
      L.bins = uint32_t((uint64_t(g->n) + (1u << bits) - 1) >> bits);
      // Parts of 1/32 of the vertices, 512 KB to 4 MB of contributions
      // (ER 4.2M: 203 us an iteration at 512 KB, 262 at 2 MB, 311 at 4 MB:
      // the blocks running together are several parts apart).
      L.part_bits = 17;
      while (L.part_bits < 20 && (uint64_t(32) << L.part_bits) < g->n) ++L.part_bits;
      L.parts = uint32_t((uint64_t(g->n) + (1u << L.part_bits) - 1) >> L.part_bits);
      const std::vector<uint32_t> &off = in->bucket_off_host;
      std::vector<uint32_t> c0(size_t(L.bins) + 1);
      uint64_t c = 0;
      for (uint32_t b = 0; b < L.bins; ++b) {
        c0[b] = uint32_t(c);
        const uint32_t v0 = b << bits;
        const uint32_t v1 = uint32_t(std::min<uint64_t>(uint64_t(v0) + (1u << bits), g->n));
        c += (uint64_t(off[v1] - off[v0]) + kChunkBuckets - 1) / kChunkBuckets;
      }
      c0[L.bins] = uint32_t(c);
      L.chunks = uint32_t(c);
      if (c * L.parts >= 0x7FFFFFFFull) return false;  // the scan counts in int
      const size_t acc_bytes = size_t(g->n) * 8 + size_t(L.bins) * 8 + 64;
      if (plan_chunk0.ensure(c0.size() * 4) || plan_cell.ensure((c * L.parts + 1) * 16) ||
          plan_acc.ensure(acc_bytes)) {
        (void)hipGetLastError();
        return false;
      }
      if (hipMemcpyAsync(plan_chunk0.ptr, c0.data(), c0.size() * 4, hipMemcpyHostToDevice,
                         stream) != hipSuccess ||
          hipStreamSynchronize(stream) != hipSuccess)
        return false;
      fill_u64(plan_acc.as<uint64_t>(), 0ull, acc_bytes / 8, stream);
      L.bin_chunk0 = plan_chunk0.as<uint32_t>();
      L.count = plan_cell.as<unsigned long long>();
      L.cell = L.count + c * L.parts + 1;
      L.acc = plan_acc.as<double>();
      L.arrived = reinterpret_cast<uint32_t *>(L.acc + g->n);
      L.bin_items = L.arrived + L.bins;
      L.n_items = L.bin_items + L.bins;
      plan = L;
    }
    const size_t cells = size_t(plan.chunks) * plan.parts;
    const unsigned pgrid = blocks_for_waves(
        std::min<uint64_t>(plan.chunks, uint64_t(device_cus(g->device)) * 32));
    fill_u64(reinterpret_cast<uint64_t *>(plan.count) + cells, 0ull, 1, stream);
    {
      ProfScope prof(stream, "k_pr_pack", 256.0 * double(in->total_buckets));
      if (in->weighted) k_pr_pack<true, false><<<pgrid, kBlock, 0, stream>>>(R, plan);
      else k_pr_pack<false, false><<<pgrid, kBlock, 0, stream>>>(R, plan);
    }
    size_t tmp = 0;
    if (hipcub::DeviceScan::ExclusiveSum(nullptr, tmp, plan.count, plan.cell, int(cells + 1),
                                         stream) != hipSuccess ||
        plan_scan.ensure(tmp)) {
      (void)hipGetLastError();
      return false;
    }
    if (hipcub::DeviceScan::ExclusiveSum(plan_scan.ptr, tmp, plan.count, plan.cell, int(cells + 1),
                                         stream) != hipSuccess ||
        hipMemcpyAsync(host.ptr, plan.cell + cells, 8, hipMemcpyDeviceToHost, stream) !=
            hipSuccess ||
        hipStreamSynchronize(stream) != hipSuccess)
      return false;
    const uint64_t m = *host.as<uint64_t>();
    // Bins of more than 9/8 of an average one are cut into items: uniform
    // graphs keep one item a bin (splitting them costs up to 1.9x), RMAT's
    // heavy bins spread over the device.
    const uint64_t cap = std::max<uint64_t>(8192, m / plan.bins + m / plan.bins / 8);
    const uint64_t most = uint64_t(plan.bins) + m / cap + 1;
    // an eighth to spare, so that growing graphs do not allocate at each call;
    // k_pr_iterate_bins reads four words at a time, the last ones included
    const uint64_t word_bytes = (m + 3) / 4 * 16;
    if ((plan_words.bytes < word_bytes && plan_words.ensure((m + m / 8 + 64) * 4)) ||
        (plan_items.bytes < most * 8 && plan_items.ensure((most + most / 8) * 8))) {
      (void)hipGetLastError();
      return false;
    }
    plan.words = plan_words.as<uint32_t>();
    plan.items = plan_items.as<uint2>();
    {
      ProfScope prof(stream, "k_pr_pack", 256.0 * double(in->total_buckets) + 4.0 * double(m));
      if (in->weighted) k_pr_pack<true, true><<<pgrid, kBlock, 0, stream>>>(R, plan);
      else k_pr_pack<false, true><<<pgrid, kBlock, 0, stream>>>(R, plan);
    }
    k_pr_items<<<1, kPlanBlock, 0, stream>>>(plan, uint32_t(std::min<uint64_t>(cap, 0xFFFFFFFFull)));
    grid = unsigned(most);
    return hipGetLastError() == hipSuccess;
  }

  int compute(float *ms) {
    MK_HIP(hipSetDevice(g->device));
    MK_HIP(hipEventRecord(ev0, stream));
    k_pr_reset<<<1, kSlots, 0, stream>>>(st);
    const PrView P = view();
    const GraphView R = in->view();
    k_pr_prepare<<<blocks_for_threads(g->n), kBlock, 0, stream>>>(P, cur);
    const unsigned grid = blocks_for_waves(
        std::min<uint64_t>((uint64_t(g->n) + 63) / 64 + hub_items / 64 + 1, uint64_t(max_waves)));
    const unsigned hgrid = blocks_for_threads(std::max<uint32_t>(n_hubs, 1));
    // The first iteration walks the slabs (ER 4.2M x 33.5M: 0.51 ms).
    // Packing costs 0.67 ms there and an iteration over the packed words
    // 0.2 ms, so it pays from the third packed iteration on: the call packs
    // unless the delta after the first says that the second is its last.
    // Whole calls (insert + delete batch, each with its iterations): ER 5k
    // 1.03 -> 0.54 ms, RMAT 40k 2.41 -> 0.79, RMAT 4.2M 34.1 -> 14.5.
    const bool may_pack = plan_fits();
    bool packed = false;
    unsigned bgrid = 0;
    uint32_t i = 0, group = may_pack ? 1 : 8;
    for (;;) {
      for (uint32_t k = 0; k < group; ++k, ++i) {
        if (packed) {
          ProfScope prof(stream, "k_pr_iterate", 4.0 * edge_estimate * 2 + 20.0 * double(g->n));
          k_pr_iterate_bins<<<bgrid, kPlanBlock, 0, stream>>>(P, plan, cur, i);
          continue;
        }
        // bytes: 256 per in-slab + 4 per key (contribution gather) and 20 per
        // vertex (bucket range, old rank, new rank, outdeg, contribution),
        // accounted with the in-adjacency size below
        ProfScope prof(stream, "k_pr_iterate", iter_bytes());
        if (in->weighted)
          k_pr_iterate<true><<<grid, kBlock, 0, stream>>>(R, P, cur, i);
        else
          k_pr_iterate<false><<<grid, kBlock, 0, stream>>>(R, P, cur, i);
        if (n_hubs) k_pr_hubs<<<hgrid, kBlock, 0, stream>>>(P, cur, i);
      }
      // a call that needs one iteration ends with this wait, not after the
      // next eight launches and another (ranks that still hold: ER 64 to 65k
      // vertices 0.113 -> 0.060 ms, RMAT-20 0.40 -> 0.32)
      if (may_pack && i == 1) k_pr_ended<<<1, 64, 0, stream>>>(P, i);
      MK_HIP(hipGetLastError());
      MK_HIP(hipMemcpyAsync(host.ptr, st, sizeof(PrState), hipMemcpyDeviceToHost, stream));
      MK_HIP(hipStreamSynchronize(stream));
      const PrState &h = *host.as<PrState>();
      if (h.stopped || h.iters < i || i >= max_iter) {
        last_iters = h.iters;
        double d = 0.0;
        if (h.iters > 0)
          for (uint32_t k = 0; k < kSlots; ++k) d += h.delta[(h.iters - 1) % 3][k];
        last_delta = d;
        break;
      }
      if (may_pack && i == 1) {
        double d = 0.0;
        for (uint32_t k = 0; k < kSlots; ++k) d += h.delta[0][k];
        if (d * double(damping) > P.margin && max_iter > 2) packed = build_plan(bgrid);
      }
      group = 8;
    }
    cur = (cur + last_iters) & 1u;
    MK_HIP(hipEventRecord(ev1, stream));
    MK_HIP(hipEventSynchronize(ev1));
    float t = 0.f;
    MK_HIP(hipEventElapsedTime(&t, ev0, ev1));
    if (ms) *ms = t;
    return MK_OK;
  }

  double iter_bytes() const {
    // in-slabs (heads + overflow are read once), one 4 B gather per edge and
    // 20 B per vertex; the edge count is the live out-degree total
    return 256.0 * double(in->total_buckets) + 20.0 * double(g->n) + 4.0 * edge_estimate;
  }
  double edge_estimate = 0.0;

  int batch(const uint32_t *src, const uint32_t *dst, uint32_t n, int sign, float *ms) {
    if (n && (!src || !dst)) return fail(MK_ERR_BAD_ARG, "pagerank: NULL batch");
    MK_HIP(hipSetDevice(g->device));
    if (n) {
      if (exact_outdeg) {
        MK_HIP(hipMemcpyAsync(outdeg, g->vdeg, size_t(g->n) * 4, hipMemcpyDeviceToDevice,
                              stream));
      } else {
        // the reverse graph saw (dst, src); use its per-edge status when this
        // is the batch it last applied, else recount from the in-adjacency
        const int op = sign > 0 ? 1 : 2;
        const bool same = g->last_op == op && g->status_n == n &&
                          ((g->last_src == dst && g->last_dst == src) ||
                           (g->last_src == src && g->last_dst == dst));
        if (same) {
          k_pr_fix_outdeg<<<blocks_for_threads(n), kBlock, 0, stream>>>(
              outdeg, src, g->status.as<uint8_t>(), n, sign);
          MK_HIP(hipGetLastError());
        } else if (int r = recount()) {
          return r;
        }
      }
    }
    return compute(ms);
  }

  int read(float *out) {
    MK_HIP(hipSetDevice(g->device));
    return read_words(reinterpret_cast<uint32_t *>(out), g->n, g->device, stream,
                      WordsOf{reinterpret_cast<const uint32_t *>(pr[cur])});
  }
};

}  // namespace mk

struct mk_pagerank {
  mk::PageRank p;
};

using namespace mk;

extern "C" {

int mk_pagerank_create(mk_graph *g, float damping, float error_margin, uint32_t max_iter,
                       const uint32_t *host_outdeg, mk_pagerank **out) {
  if (!out) return fail(MK_ERR_BAD_ARG, "mk_pagerank_create: out is NULL");
  *out = nullptr;
  if (!g) return fail(MK_ERR_BAD_ARG, "mk_pagerank_create: NULL graph");
  if (!(damping >= 0.f && damping < 1.f)) return fail(MK_ERR_BAD_ARG, "damping must be in [0, 1)");
  if (!(error_margin >= 0.f)) return fail(MK_ERR_BAD_ARG, "error margin must be >= 0");
  mk_pagerank *h = new mk_pagerank();
  int r = h->p.init(g, damping, error_margin, max_iter, host_outdeg);
  if (r) {
    h->p.destroy();
    delete h;
    return r;
  }
  uint64_t m = 0;
  if (mk_graph_num_edges(g, &m) == MK_OK) h->p.edge_estimate = double(m);
  g->users++;
  *out = h;
  return MK_OK;
}

int mk_pagerank_destroy(mk_pagerank *p) {
  if (!p) return fail(MK_ERR_BAD_ARG, "mk_pagerank_destroy: NULL handle");
  p->p.g->users--;
  p->p.destroy();
  delete p;
  return MK_OK;
}

int mk_pagerank_static(mk_pagerank *p, float *ms) {
  if (!p) return fail(MK_ERR_BAD_ARG, "mk_pagerank_static: NULL handle");
  if (int r = graph_settle(p->p.g)) return r;
  return p->p.compute(ms);
}

int mk_pagerank_incremental(mk_pagerank *p, const uint32_t *src, const uint32_t *dst, uint32_t n,
                            float *ms) {
  if (!p) return fail(MK_ERR_BAD_ARG, "mk_pagerank_incremental: NULL handle");
  if (int r = graph_settle(p->p.g)) return r;
  // a graph of reversed edges saw the batch as (dst, src)
  if (int r = graph_failed_batch(p->p.g, src, dst, n)) return r;
  if (int r = graph_failed_batch(p->p.g, dst, src, n)) return r;
  return p->p.batch(src, dst, n, +1, ms);
}

int mk_pagerank_decremental(mk_pagerank *p, const uint32_t *src, const uint32_t *dst, uint32_t n,
                            float *ms) {
  if (!p) return fail(MK_ERR_BAD_ARG, "mk_pagerank_decremental: NULL handle");
  if (int r = graph_settle(p->p.g)) return r;
  if (int r = graph_failed_batch(p->p.g, src, dst, n)) return r;
  if (int r = graph_failed_batch(p->p.g, dst, src, n)) return r;
  return p->p.batch(src, dst, n, -1, ms);
}

int mk_pagerank_read(mk_pagerank *p, float *values) {
  if (!p || !values) return fail(MK_ERR_BAD_ARG, "mk_pagerank_read: NULL argument");
  return p->p.read(values);
}

int mk_pagerank_last_stats(mk_pagerank *p, uint32_t *iterations, double *last_delta) {
  if (!p) return fail(MK_ERR_BAD_ARG, "mk_pagerank_last_stats: NULL handle");
  if (iterations) *iterations = p->p.last_iters;
  if (last_delta) *last_delta = p->p.last_delta;
  return MK_OK;
}

}  // extern "C"
