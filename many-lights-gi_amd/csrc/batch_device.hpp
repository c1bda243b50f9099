// Device helpers of the batched kernels (one launch per stage over all frames
// of a batch).
#pragma once

#include "kernels.hpp"

namespace mlgi {

// Frame of the batch whose range of one stage's items holds `item`: the last
// frame with first <= item (frames are sorted by that stage's first item).
template <uint32_t BatchFrame::*kFirst>
__device__ __forceinline__ int batch_find(const BatchFrame* __restrict__ f, int n, uint32_t item) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (f[mid].*kFirst <= item)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

// Loads and stores through global-address-space pointers. Pointers read from
// a frame table (or any struct in memory) are generic, and generic accesses
// compile to flat instructions, which count against both the vector-memory
// and the LDS wait counters: every LDS wait then also waits for outstanding
// global loads. These helpers make such accesses global_load / global_store.
template <class T>
__device__ __forceinline__ T gload(const T* p) {
  return *(const __attribute__((address_space(1))) T*)p;
}
// 16-byte loads: through the native vector type (the HIP vector class would
// be copied through a generic reference, which is flat again).
__device__ __forceinline__ float4 gload4(const float4* p) {
  typedef float v4f __attribute__((ext_vector_type(4)));
  const v4f v = *(const __attribute__((address_space(1))) v4f*)p;
  return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint4 gload4(const uint4* p) {
  typedef unsigned int v4u __attribute__((ext_vector_type(4)));
  const v4u v = *(const __attribute__((address_space(1))) v4u*)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}
// Relaxed, agent-scope atomics on global memory (no return value needed
// except for the add).
__device__ __forceinline__ uint32_t gatomic_add(uint32_t* p, uint32_t v) {
  return __hip_atomic_fetch_add((__attribute__((address_space(1))) uint32_t*)p, v, __ATOMIC_RELAXED,
                                __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void gatomic_min(uint32_t* p, uint32_t v) {
  (void)__hip_atomic_fetch_min((__attribute__((address_space(1))) uint32_t*)p, v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void gatomic_or(uint32_t* p, uint32_t v) {
  (void)__hip_atomic_fetch_or((__attribute__((address_space(1))) uint32_t*)p, v, __ATOMIC_RELAXED,
                              __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void gstore(T* p, T v) {
  *(__attribute__((address_space(1))) T*)p = v;
}

constexpr int kBatchXcds = 8;

// Item of workgroup blockIdx.x in a launch of one workgroup per item over a
// grid of xcd_items_grid(items) workgroups. Workgroups are dispatched to the
// XCDs round robin, so workgroup b runs on XCD b mod 8; the items are dealt to
// the XCDs in chunks of consecutive ones, which share inputs (neighbouring
// ISMs and bins) through one L2, chunk c to XCD c mod 8. Items at or past
// `items` have no work.
//
// Chunks of 32 (fewer where that leaves an XCD under four of them): one
// contiguous eighth per XCD gave a batch's XCDs whole frames, and a frame of
// 256 bins holds as many points as one of 4,096, so the XCD with the small
// frames worked while the others were done. 16 frames of 256..4,096 VPLs and
// 1M points each: tiles 731 us and masks 211 with contiguous eighths, 310 and
// 129 with chunks of 256, 267 and 113 with 64, 259 and 108 with 32, 277 and
// 108 with 4. One frame: 1080p tiles 30.0 (eighths), 29.4 (32), 30.2 (4); 4K
// 99.8, 97.7, 103.0.
__host__ __device__ inline uint32_t xcd_chunk_log2(uint32_t items) {
  const uint32_t l = 31u - (uint32_t)__builtin_clz(items | 32u);  // floor(log2), at least 5
  return l > 10u ? 5u : l - 5u;
}
__device__ __forceinline__ uint32_t xcd_item(uint32_t items) {
  const uint32_t l = xcd_chunk_log2(items);
  const uint32_t xcd = blockIdx.x % kBatchXcds, i = blockIdx.x / kBatchXcds;
  return (((i >> l) * kBatchXcds + xcd) << l) | (i & ((1u << l) - 1u));
}
inline unsigned xcd_items_grid(uint32_t items) {
  const uint64_t round = (uint64_t)kBatchXcds << xcd_chunk_log2(items);
  return (unsigned)((items + round - 1) / round * round);
}

}  // namespace mlgi
