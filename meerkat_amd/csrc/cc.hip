// Connected components by concurrent union-find over the slab-hash graph.
//
// Reference: include/Util/UnionFind.cuh (primitives only; no caller and no
// CC driver in the reference).  UnionAsync (:122-149) finds both roots and
// links the larger root under the smaller with atomicCAS; this keeps every
// parent pointer <= its vertex, so a component's root is its smallest vertex
// and the labels are canonical (min vertex id) with no relabelling pass.
// Find uses path halving with plain stores (find_op::FindCompress / halving
// variants, :24-86): a halving store only replaces a parent by one of its
// ancestors, which keeps parent[x] <= x, so concurrent halving is safe.
//
// Edges are taken as undirected (weak components).  Static = union over one
// or two edges of every vertex, a compress pass (label = root), union over
// the edges in the slabs whose ends' labels still differ (the sampling of
// Sutton, Ben-Nun and Barak, "Optimizing parallel graph connectivity
// computation via subgraph sampling", IPDPS 2018; every edge is looked at,
// since a graph may hold an edge in one direction only), compress again.  Incremental
// = union over the inserted batch, then compress.  Decremental recomputes
// (union-find cannot split components).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "profile.hpp"
#include "readback.hpp"
#include "slabhash.hpp"

namespace mk {

MK_DEV uint32_t uf_find(uint32_t *parent, uint32_t x) {
  uint32_t p = parent[x];
  while (p != x) {
    const uint32_t gp = parent[p];
    if (gp != p) parent[x] = gp;  // halving: gp is an ancestor, gp <= p
    x = p;
    p = parent[x];
  }
  return x;
}

// Root of x reading parents with agent-coherent loads (no halving).
MK_DEV uint32_t uf_find_coherent(uint32_t *parent, uint32_t x) {
  for (;;) {
    const uint32_t p = coherent_load(parent + x);
    if (p == x) return x;
    x = p;
  }
}

// Link the roots of a and b, the larger under the smaller.  A plain load may
// return an older parent; older parents are still ancestors (pointers only
// move up), so a stale walk ends at a vertex on the true path and a lost CAS
// is the only consequence.  After a lost CAS the walk resumes from the
// parent the CAS returned, with coherent loads, so every retry climbs
// strictly and the loop ends.
MK_DEV void uf_union(uint32_t *parent, uint32_t a, uint32_t b) {
  bool fresh = false;
  for (;;) {
    uint32_t ra = fresh ? uf_find_coherent(parent, a) : uf_find(parent, a);
    uint32_t rb = fresh ? uf_find_coherent(parent, b) : uf_find(parent, b);
    if (ra == rb) return;
    if (ra < rb) {
      const uint32_t t = ra;
      ra = rb;
      rb = t;
    }
    // ra > rb: hang ra under rb if ra is still a root
    const uint32_t old = atomicCAS(parent + ra, ra, rb);
    if (old == ra) return;
    a = old;  // ra's current parent (smaller than ra)
    b = rb;
    fresh = true;
  }
}

// Sampling steps before the edge pass.  Whole static passes, against finds
// for both ends of every edge: RMAT-21 1.79 -> 0.67 ms, RMAT-18 0.64 -> 0.10,
// ER 1M x 16M 0.75 -> 0.52, ER 1M x 1M 0.57 -> 0.30, a path of 1M vertices
// 0.90 -> 0.14, a grid of 1M 0.69 -> 0.15.
constexpr uint32_t kSampleSteps = 4;
constexpr uint32_t kHookBlock = 1024;
// The last step runs where kManyApart of kAsked vertices, spread over the
// graph, still have a sampled key of another label: sparse uniform graphs,
// whose trees join step by step, not RMAT ones, whose hubs have joined nearly
// all.  Where many edges are left to k_cc_edges their unions meet on few
// roots: weighted ER 131k x 1M took 2.0 ms with two keys a step (0.16 without
// sampling, 0.12 now), ER 131k x 262k 0.65 without the last step (0.19, 0.11).
// Small graphs leave few edges in any case, and the launches are a fifth of
// their call (RMAT-14: 40 us with, 34 without).
constexpr uint32_t kAsked = 1u << 14;
constexpr uint32_t kManyApart = kAsked / 64;
constexpr uint32_t kFewVertices = 1u << 15;

__global__ void k_cc_init(uint32_t *parent, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) parent[i] = i;
}

// Four keys of vertex u in one line of its first slab: words `word`, +1, +16
// and +17, of a map +0, +2, +16 and +18.  Inserts fill words 0, (1,) 16,
// (17,) 32, (33,) 48, (49,) first, then 2, ....  kEmpty: none.
template <bool MAP> MK_DEV void first_keys(const GraphView &G, uint32_t u, uint32_t word,
                                           uint32_t (&k)[4]) {
  const uint32_t *slab = G.heads + size_t(G.bucket_off[u]) * kSlabWords + word;
  if (MAP) {
    const uint4 a = *reinterpret_cast<const uint4 *>(slab);
    const uint4 b = *reinterpret_cast<const uint4 *>(slab + 16);
    k[0] = a.x;
    k[1] = a.z;
    k[2] = b.x;
    k[3] = b.z;
  } else {
    const uint2 a = *reinterpret_cast<const uint2 *>(slab);
    const uint2 b = *reinterpret_cast<const uint2 *>(slab + 16);
    k[0] = a.x;
    k[1] = a.y;
    k[2] = b.x;
    k[3] = b.y;
  }
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q)
    if (k[q] >= kTomb) k[q] = kEmpty;
}

// Sampling step 0: every vertex hangs under the smallest of itself and its
// first keys (a forest: parents are smaller); parents within the block's
// vertices are followed in LDS right away, so that neighbours in id order
// (paths, grids) make no long chains for the compress pass.
template <bool MAP>
__global__ void __launch_bounds__(kHookBlock)
    k_cc_hook(GraphView G, uint32_t *parent, uint32_t *apart) {
  __shared__ uint32_t lp[kHookBlock];
  const uint32_t t = threadIdx.x, base = blockIdx.x * kHookBlock, u = base + t;
  if (u == 0) *apart = 0u;
  uint32_t p = u;
  if (u < G.n && G.vdeg[u] != 0) {
    uint32_t k[4];
    first_keys<MAP>(G, u, 0, k);
    p = min(min(min(k[0], k[1]), min(k[2], k[3])), u);
  }
#pragma unroll 1
  for (uint32_t len = 1; len < kHookBlock; len <<= 1) {  // pointer doubling
    lp[t] = p;
    __syncthreads();
    if (p >= base) p = lp[p - base];
    __syncthreads();
  }
  if (u < G.n) parent[u] = p;
}

// Sampling steps 1, 2, ..., paths shortened in between: the vertex's label
// (a root, mostly) takes the smallest label among its keys in words `word`, if that
// is smaller.  Of several offers to one root the smallest stays; the edges
// of the others join in a later step or in k_cc_edges.  No step waits or
// retries: finds and CAS loops from every vertex at once made chains that
// took 0.3 ms on RMAT-21 and 8 ms on a path of 1M vertices.  With `apart`
// (k_cc_ask's count), nothing unless there are many.
template <bool MAP>
__global__ void k_cc_sample(GraphView G, uint32_t *parent, uint32_t word,
                            const uint32_t *apart) {
  if (apart && *apart < kManyApart) return;
  const uint32_t u = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t pu = 0, lo = 0;
  if (u < G.n && G.vdeg[u] != 0) {
    uint32_t k[4];
    first_keys<MAP>(G, u, word, k);
    lo = pu = parent[u];
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q)
      if (k[q] != kEmpty) lo = min(lo, parent[k[q]]);
  }
  bool offer = lo < pu;
  uint64_t m = ballot(offer);
  // two labels' offers go out once a wave: a large tree's vertices all have
  // one for it, and accesses to one line follow one another (ER 131k x 1M,
  // sorted: 0.40 -> 0.13 ms)
  for (uint32_t t = 0; t < 2 && m; ++t) {
    const uint32_t j = ffs64(m), label = read_lane(pu, j);
    const bool same = offer && pu == label;
    uint32_t best = same ? lo : kEmpty;
#pragma unroll
    for (uint32_t o = 32; o >= 1; o >>= 1)
      best = min(best, uint32_t(__shfl_xor(int(best), int(o), 64)));
    if (lane_id() == j && coherent_load(parent + label) > best) atomicMin(parent + label, best);
    offer = offer && !same;
    m = ballot(offer);
  }
  if (offer && coherent_load(parent + pu) > lo) atomicMin(parent + pu, lo);
}

// Of kAsked vertices, those with a sampled key of another label.
template <bool MAP>
__global__ void k_cc_ask(GraphView G, const uint32_t *parent, uint32_t *apart) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t u = uint32_t(uint64_t(i) * G.n / kAsked);
  bool differs = false;
  if (i < kAsked && G.vdeg[u] != 0) {
    uint32_t k[4];
    first_keys<MAP>(G, u, 0, k);
    const uint32_t pu = parent[u];
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q)
      if (k[q] != kEmpty) differs |= parent[k[q]] != pu;
  }
  const uint64_t m = ballot(differs);
  if (m && lane_id() == 0) atomicAdd(apart, uint32_t(__popcll(m)));
}

// Union over edge (u, x) whose ends had labels pu and px: nothing where one
// step up from the labels shows one component (a label that has been hung
// under another one leaves a difference to all its edges).
MK_DEV void join_labels(uint32_t *parent, uint32_t u, uint32_t x, uint32_t pu, uint32_t px) {
  const uint32_t a = parent[pu], b = parent[px];
  if (a != b && a != px && b != pu) uf_union(parent, u, x);
}

// Union over the edges whose ends have different labels: an 8-lane group per
// bucket, a slab's neighbour labels gathered together (eight slabs in flight
// per wave).  Labels were shortened to roots before, so almost every edge
// ends at that gather; equal labels always mean one component, and where
// they differ the union looks for the roots.  Bound by the gathers (4 bytes from an
// array of 4 bytes a vertex): RMAT-21, 62M stored edges, 0.43 ms.
template <bool MAP>
__global__ void __launch_bounds__(kBlock) k_cc_edges(GraphView G, uint32_t *parent) {
  const uint32_t gl = group_lane();
  const uint64_t g0 = (uint64_t(blockIdx.x) * blockDim.x + threadIdx.x) / kGroupLanes;
  const uint64_t NG = uint64_t(gridDim.x) * blockDim.x / kGroupLanes;
  for (uint64_t b = g0; b < G.total_buckets; b += NG) {
    const uint32_t u = G.bucket_owner[b];
    if (G.vdeg[u] == 0) continue;
    const uint32_t pu = parent[u];
    const uint32_t *slab = G.heads + b * kSlabWords;
    for (;;) {
      uint32_t x[kWordsPerLane], px[kWordsPerLane];
      load_words(slab + kWordsPerLane * gl, x);
#pragma unroll
      for (uint32_t k = 0; k < kWordsPerLane; ++k)
        px[k] = key_word<MAP>(kWordsPerLane * gl + k) && x[k] < kTomb ? parent[x[k]] : pu;
#pragma unroll
      for (uint32_t k = 0; k < kWordsPerLane; ++k)
        if (px[k] != pu) join_labels(parent, u, x[k], pu, px[k]);
      const uint32_t nx = group_read(x[kWordsPerLane - 1], kGroupLanes - 1);
      if (nx == kEmpty) break;
      slab = slab_ptr(G.pool, nx);
    }
  }
}

// Union over a batch of edges (thread per edge).
__global__ void k_cc_batch(uint32_t *parent, const uint32_t *src, const uint32_t *dst,
                           uint32_t n, uint32_t nv) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t u = src[i], v = dst[i];
  if (u != v && u < nv && v < nv) uf_union(parent, u, v);
}

// label = root: every parent pointer jumps to its root.
__global__ void k_cc_compress(uint32_t *parent, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t r = parent[i];
  while (parent[r] != r) r = parent[r];
  parent[i] = r;
}

// The same between sampling steps, halving paths on the way, so that the
// threads of a long chain shorten it together.  A halving store may land
// after another thread's and leave an ancestor that is not the root: no
// harm to the steps that follow, but labels end with k_cc_compress.
__global__ void k_cc_shorten(uint32_t *parent, uint32_t n, const uint32_t *apart) {
  if (apart && *apart < kManyApart) return;
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) parent[i] = uf_find(parent, i);
}

struct CC {
  mk_graph *g = nullptr;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  uint32_t *parent = nullptr;  // n parents (labels), then k_cc_ask's count

  int init(mk_graph *graph) {
    g = graph;
    MK_HIP(hipSetDevice(g->device));
    MK_HIP(hipStreamCreate(&stream));
    loop_stream_add(g->device, stream, 1);
    MK_HIP(hipEventCreate(&ev0));
    MK_HIP(hipEventCreate(&ev1));
    MK_HIP(hipMalloc(&parent, (size_t(g->n) + 1) * 4));
    k_cc_init<<<blocks_for_threads(g->n), kBlock, 0, stream>>>(parent, g->n);
    MK_HIP(hipStreamSynchronize(stream));
    return MK_OK;
  }

  void destroy() {
    (void)hipSetDevice(g->device);
    if (stream) (void)hipStreamSynchronize(stream);
    (void)hipFree(parent);
    if (ev0) (void)hipEventDestroy(ev0);
    if (ev1) (void)hipEventDestroy(ev1);
    if (stream) {
      loop_stream_add(g->device, stream, -1);
      (void)hipStreamDestroy(stream);
    }
  }

  int finish(float *ms) {
    {
      // per vertex: parent read + root read + write
      ProfScope prof(stream, "k_cc_compress", 12.0 * g->n);
      k_cc_compress<<<blocks_for_threads(g->n), kBlock, 0, stream>>>(parent, g->n);
    }
    MK_HIP(hipGetLastError());
    MK_HIP(hipEventRecord(ev1, stream));
    MK_HIP(hipEventSynchronize(ev1));
    float t = 0.f;
    MK_HIP(hipEventElapsedTime(&t, ev0, ev1));
    if (ms) *ms = t;
    return MK_OK;
  }

  int run_static(float *ms) {
    MK_HIP(hipSetDevice(g->device));
    MK_HIP(hipEventRecord(ev0, stream));
    const unsigned grid = blocks_for_waves(std::min<uint64_t>(
        (uint64_t(g->total_buckets) + 7) / 8, uint64_t(device_cus(g->device)) * 32));
    {
      // per vertex: degree, bucket, first words, two labels
      ProfScope prof(stream, "k_cc_sample", kSampleSteps * 40.0 * g->n);
      auto hook = g->weighted ? k_cc_hook<true> : k_cc_hook<false>;
      auto sample = g->weighted ? k_cc_sample<true> : k_cc_sample<false>;
      auto ask = g->weighted ? k_cc_ask<true> : k_cc_ask<false>;
      uint32_t *apart = parent + g->n;
      const uint32_t steps = g->n > kFewVertices ? kSampleSteps : kSampleSteps - 1;
      for (uint32_t step = 0; step < steps; ++step) {
        const uint32_t *when = step == kSampleSteps - 1 ? apart : nullptr;
        if (when) ask<<<kAsked / kBlock, kBlock, 0, stream>>>(g->view(), parent, apart);
        if (step == 0)
          hook<<<unsigned((uint64_t(g->n) + kHookBlock - 1) / kHookBlock), kHookBlock, 0,
                 stream>>>(g->view(), parent, apart);
        else
          sample<<<blocks_for_threads(g->n), kBlock, 0, stream>>>(g->view(), parent,
                                                                  step == 2 ? 32 : 0, when);
        k_cc_shorten<<<blocks_for_threads(g->n), kBlock, 0, stream>>>(parent, g->n, when);
      }
    }
    {
      // per bucket: owner + degree (8 B) and its slabs; per edge one label
      uint64_t m = 0;
      if (profiling_on()) (void)mk_graph_num_edges(g, &m);
      ProfScope prof(stream, "k_cc_edges", 264.0 * g->total_buckets + 4.0 * double(m));
      if (g->weighted)
        k_cc_edges<true><<<grid, kBlock, 0, stream>>>(g->view(), parent);
      else
        k_cc_edges<false><<<grid, kBlock, 0, stream>>>(g->view(), parent);
    }
    MK_HIP(hipGetLastError());
    return finish(ms);
  }

  int run_incremental(const uint32_t *src, const uint32_t *dst, uint32_t n, float *ms) {
    if (n && (!src || !dst)) return fail(MK_ERR_BAD_ARG, "cc incremental: NULL batch");
    MK_HIP(hipSetDevice(g->device));
    MK_HIP(hipEventRecord(ev0, stream));
    if (n) {
      ProfScope prof(stream, "k_cc_batch", 20.0 * n);
      k_cc_batch<<<blocks_for_threads(n), kBlock, 0, stream>>>(parent, src, dst, n, g->n);
    }
    MK_HIP(hipGetLastError());
    return finish(ms);
  }
};

}  // namespace mk

struct mk_cc {
  mk::CC c;
};

using namespace mk;

extern "C" {

int mk_cc_create(mk_graph *g, mk_cc **out) {
  if (!out) return fail(MK_ERR_BAD_ARG, "mk_cc_create: out is NULL");
  *out = nullptr;
  if (!g) return fail(MK_ERR_BAD_ARG, "mk_cc_create: NULL graph");
  mk_cc *h = new mk_cc();
  int r = h->c.init(g);
  if (r) {
    h->c.destroy();
    delete h;
    return r;
  }
  g->users++;
  *out = h;
  return MK_OK;
}

int mk_cc_destroy(mk_cc *c) {
  if (!c) return fail(MK_ERR_BAD_ARG, "mk_cc_destroy: NULL handle");
  c->c.g->users--;
  c->c.destroy();
  delete c;
  return MK_OK;
}

int mk_cc_static(mk_cc *c, float *ms) {
  if (!c) return fail(MK_ERR_BAD_ARG, "mk_cc_static: NULL handle");
  if (int r = graph_settle(c->c.g)) return r;
  return c->c.run_static(ms);
}

int mk_cc_incremental(mk_cc *c, const uint32_t *src, const uint32_t *dst, uint32_t n,
                      float *ms) {
  if (!c) return fail(MK_ERR_BAD_ARG, "mk_cc_incremental: NULL handle");
  if (int r = graph_settle(c->c.g)) return r;
  if (int r = graph_failed_batch(c->c.g, src, dst, n)) return r;
  return c->c.run_incremental(src, dst, n, ms);
}

int mk_cc_decremental(mk_cc *c, const uint32_t *src, const uint32_t *dst, uint32_t n,
                      float *ms) {
  (void)src;
  (void)dst;
  (void)n;
  if (!c) return fail(MK_ERR_BAD_ARG, "mk_cc_decremental: NULL handle");
  if (int r = graph_settle(c->c.g)) return r;
  return c->c.run_static(ms);
}

int mk_cc_labels(mk_cc *c, uint32_t *labels) {
  if (!c || !labels) return fail(MK_ERR_BAD_ARG, "mk_cc_labels: NULL argument");
  MK_HIP(hipSetDevice(c->c.g->device));
  return read_words(labels, c->c.g->n, c->c.g->device, c->c.stream, WordsOf{c->c.parent});
}

}  // extern "C"
