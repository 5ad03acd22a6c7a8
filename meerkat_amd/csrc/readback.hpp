// Results to host memory.
//
// A caller's result array is ordinary (pageable) host memory, usually fresh:
// hipMemcpy into it stages through the runtime's own buffers on one thread
// at 10 GB/s on MI355X (17 GB/s once the pages exist), where the link does
// 56 GB/s.  Here a kernel writes 1 MB chunks of the result straight into
// pinned host memory, in its final form (no device copy of the result), and
// up to kReadSlots threads, one per slot, copy them on, so that link,
// copying and the first touch of the caller's pages overlap.  The pinned
// memory (8 MB for each of up to kReadStages readers at a time) is shared by
// all handles; it is allocated by the first reads and freed with the last
// slab pool.
#pragma once

#include <functional>

#include "mk_internal.hpp"

namespace mk {

constexpr uint32_t kReadWords = 1u << 18;  // words per chunk
constexpr uint32_t kReadSlots = 8;
constexpr uint32_t kReadStages = 4;
constexpr uint32_t kReadBlocks = 32;       // blocks per chunk, a flag word each
constexpr uint32_t kReadThreads = 1024;

// What is read: word i of the result.
struct WordsOf {
  const uint32_t *p;
  MK_DEV uint32_t operator()(size_t i) const { return p[i]; }
};
struct HighOf {
  const uint64_t *p;
  MK_DEV uint32_t operator()(size_t i) const { return uint32_t(p[i] >> 32); }
};
struct LowOf {
  const uint64_t *p;
  MK_DEV uint32_t operator()(size_t i) const { return uint32_t(p[i]); }
};
struct ColumnOf {  // column `c` of rows of 64 words
  const uint32_t *p;
  uint32_t c;
  MK_DEV uint32_t operator()(size_t i) const { return p[i * 64 + c]; }
};

// Words [first, first + count) of f into `dst` (pinned host memory, device
// alias, kReadWords long; or device memory with flags == nullptr).  Stores
// are system-scope, so once a wave's have completed (vmcnt 0) the host sees
// them; each block then writes `seq` into its flag.
template <typename F>
__global__ void __launch_bounds__(kReadThreads)
    k_read_chunk(F f, uint32_t *dst, size_t first, uint32_t count, uint32_t *flags, uint32_t seq) {
#pragma unroll 4
  for (uint32_t i = (blockIdx.x * kReadThreads + threadIdx.x) * 2; i < count;
       i += kReadBlocks * kReadThreads * 2) {
    const uint32_t a = f(first + i);
    const uint32_t b = i + 1 < count ? f(first + i + 1) : 0u;
    if (flags)
      __hip_atomic_store(reinterpret_cast<uint64_t *>(dst + i), (uint64_t(b) << 32) | a,
                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else
      *reinterpret_cast<uint64_t *>(dst + i) = (uint64_t(b) << 32) | a;
  }
  if (!flags) return;
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(flags + blockIdx.x, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

using ReadLaunch =
    std::function<void(uint32_t *dst, size_t first, uint32_t count, uint32_t *flags, uint32_t seq)>;
// Read `words` words, chunk by chunk, launched by `launch` on stream `s`
// (graph.hip); returns when they are in `out`.
int read_chunks(uint32_t *out, size_t words, int device, hipStream_t s, const ReadLaunch &launch);

// `words` words of f into host memory `out`, after the work queued on `s`.
template <typename F>
int read_words(uint32_t *out, size_t words, int device, hipStream_t s, F f) {
  return read_chunks(out, words, device, s,
                     [=](uint32_t *dst, size_t first, uint32_t count, uint32_t *flags,
                         uint32_t seq) {
                       k_read_chunk<F><<<kReadBlocks, kReadThreads, 0, s>>>(f, dst, first, count,
                                                                           flags, seq);
                     });
}

}  // namespace mk
