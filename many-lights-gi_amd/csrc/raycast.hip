// Device G-buffer / RSM producer: the scene's BVH ray cast on the GPU.
// Replaces the reference's rasterisation of the G-buffer and RSM
// (RasterizationStage.cpp and model.frag) for inputs that change per request
// or per frame. Rays, triangle tests and shading are the host renderer's
// double-precision code (scene_trace.hpp, compiled with -ffp-contract=off
// like it), and which triangle wins does not depend on the order of the
// visits, so both write the same texels.
//
// What bounds it. One traversal per lane spends its time on divergence (an
// inner step and a leaf step both issue for the whole wave), on the latency
// of each step's node load, and on the LDS of 64 private stacks (six waves
// per CU). The rays of a wave's tile are so coherent, though, that one
// traversal for all of them visits hardly more nodes than one ray's: at 1080p
// and 40k triangles 23.7 nodes and 11.5 leaves per 8 x 8 tile against 20.8 and
// 8.9 per ray, for a 128^2 RSM of 160k triangles 22 and 17 per 4 x 4 tile
// against 21 and 15 (counted on the CPU). So a wave is a packet: it walks the
// 8-wide tree once, visiting a child if any of its rays enters the child's
// box before that ray's nearest hit. The current node is wave-uniform, so
// there is no divergence, and the stack holds one reference per pending child
// and one entry distance per ray.
//
// Boxes are tested in FP32 against node boxes that carry a margin for it
// (kBoxMargin), which can only visit more nodes; a packet also tests
// triangles whose box some of its rays miss. Neither changes a texel: every
// hit is decided by the exact triangle test.
//
// Two forms of a packet, in single-wave workgroups:
//   * 8 x 8 rays, one lane each, for images of 512^2 texels or more: bound by
//     VALU issue. Node and triangle data are wave-uniform and read through
//     the scalar cache; each lane tests all children of a node and all
//     triangles of a leaf for its ray.
//   * 4 x 4 rays of four lanes each for smaller images, which are bound by
//     the latency of the steps of their longest packets (a 128^2 RSM is one
//     wave per SIMD): lane q of a ray's quad tests children q and q + 4 and a
//     leaf's triangle q, a quarter of the instructions per step.
// Measured (one traversal per lane or quad over a 4-wide tree -> packets):
// 1080p G-buffer of 40k triangles 2,234 -> 423 us, 128^2 RSM of 160k
// 179 -> 61 us, 512^2 RSM 319 -> 115 us. The line between the forms: a 256^2
// G-buffer takes 77 us in the second form and 136 in the first, a 512^2 one
// 154 and 145.
#include "kernels.hpp"
#include "scene_trace.hpp"

namespace mlgi {
namespace {

using namespace mlgi_scene_impl;

constexpr size_t kWideRays = (size_t(1) << 18) - 1;

// Pending children whose entry distances are kept; deeper ones are visited
// without that test. 24 lets the 8 x 8 form run six waves per SIMD, as many as
// its registers allow (1080p G-buffer, 40k triangles: 423 us, 442 with 32
// entries); few packets have more pending (19 at most there, 26 in a 128^2
// RSM of 160k triangles).
constexpr int kNearStack = 24;

template <int kRays>
struct PacketLds {
  float near[kNearStack * kRays];
  uint32_t ref[kTraceStack];
};

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ bool any_lane(bool b) { return __ballot(b) != 0ull; }

// The packet's box rays: one that starts outside the scene's box is moved to
// its entry (the margin of the scene's box covers the double rounding here).
__device__ __forceinline__ BoxRay packet_box_ray(const SceneView& s, D3 o, D3 d, double tmax) {
  bool in = true;
  double entry = 0.0;
  const bool outside = outside_scene(s, o);
  if (any_lane(outside)) {
    double t0;
    in = box_hit(s.lo, s.hi, o, ray_inverse(d), tmax, &t0);
    if (outside && in) entry = t0;
  }
  return box_ray(o, d, entry, tmax, in);
}

// The packet's direction octant, from its first lane: any octant orders the
// visits correctly, and the rays of a packet rarely differ.
__device__ __forceinline__ int packet_octant(D3 d) {
  const int o = (d.x < 0.0 ? 1 : 0) | (d.y < 0.0 ? 2 : 0) | (d.z < 0.0 ? 4 : 0);
  return __builtin_amdgcn_readfirstlane(o);
}

// Pops the nearest pending child that some lane's ray still enters before
// its nearest hit. `slot` is the lane's ray in the packet. False when none is
// left.
template <int kRays>
__device__ __forceinline__ bool packet_pop(const PacketLds<kRays>& lds, int slot, float tmax, int& sp,
                                           uint32_t& cur) {
  wave_sync();  // the stack's entries were written by other lanes
  while (sp > 0) {
    --sp;
    const uint32_t ref = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds.ref[sp]);
    const float near = sp < kNearStack ? lds.near[sp * kRays + slot] : 0.0f;
    if (any_lane(near <= tmax)) {
      cur = ref;
      return true;
    }
  }
  return false;
}

// ---------------------------------------------------- 8 x 8 rays, a lane each

template <class T>
using Uniform = const __attribute__((address_space(4))) T;  // read through the scalar cache

__device__ Hit trace_rays(const SceneView& s, D3 o, D3 d, double tmax, PacketLds<64>& lds) {
  typedef float f8 __attribute__((ext_vector_type(8)));
  const int lane = threadIdx.x;
  Hit h{tmax, -1};
  BoxRay r = packet_box_ray(s, o, d, tmax);
  const int oct = packet_octant(d);
  const int pair = oct < 4 ? oct : oct ^ 7;  // the stored order; reversed for octants 4..7
  int sp = 0;
  uint32_t cur = 0;  // the root, an inner node
  while (true) {
    const int count = (int)(cur & 7u);
    const uint32_t first = cur >> 3;
    if (count == 0) {
      Uniform<f8>* nd = (Uniform<f8>*)(s.nodes + first);
      Uniform<uint32_t>* words = (Uniform<uint32_t>*)(s.nodes + first);
      const uint32_t after_lo = words[16 * pair + 7], after_hi = words[16 * pair + 15];
      float near[8];
      uint32_t ref[8];
      uint32_t hits = 0;
      auto test = [&](int k) {
        const f8 c = nd[k];
        ref[k] = __float_as_uint(c[6]);
        const bool hit = box_test(r, c[0], c[1], c[2], c[3], c[4], c[5], near[k]);
        if (!hit) near[k] = __builtin_inff();
        hits |= any_lane(hit) ? 1u << k : 0u;
      };
#pragma unroll
      for (int k = 0; k < 4; ++k) test(k);
      if (words[8 * 4 + 6] != kNoChild) {
#pragma unroll
        for (int k = 4; k < 8; ++k) test(k);
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (!(hits >> k & 1u)) continue;
        uint32_t after = ((k < 4 ? after_lo : after_hi) >> (8 * (k & 3))) & 0xFFu;
        if (oct >= 4) after = ~after & ~(1u << k);
        if ((hits & after) == (hits ^ 1u << k)) {  // the nearest child is visited next
          cur = ref[k];
          continue;
        }
        const int pos = sp + __builtin_popcount(hits & after);  // < kTraceStack (the build's bound)
        if (pos < kNearStack) lds.near[pos * 64 + lane] = near[k];
        if (lane == 0) lds.ref[pos] = ref[k];
      }
      if (hits != 0u) {
        sp += __builtin_popcount(hits) - 1;
        continue;
      }
    } else {
      auto load = [&](int k) {
        Uniform<double>* g = (Uniform<double>*)(s.geo + first + k);
        return TriGeo{{g[0], g[1], g[2]}, {g[3], g[4], g[5]}, {g[6], g[7], g[8]}};
      };
      TriGeo next = load(0);
      for (int k = 0; k < count; ++k) {
        const TriGeo t = next;
        next = load(k + 1);  // requested before this one is tested; padded past the last triangle
        const TriTerms q = tri_terms(t, o, d);
        const bool maybe = tri_maybe(q, h.t);
        if (any_lane(maybe)) {
          double th;
          if (maybe && tri_accept(q, h.t, &th) && hit_before(th, (int)first + k, h)) {
            h.t = th;
            h.tri = (int)first + k;
            r.tmax = box_tmax(th, r.entry);
          }
        }
      }
    }
    if (!packet_pop(lds, lane, r.tmax, sp, cur)) break;
  }
  if (h.tri >= 0) h.tri = s.order[h.tri];
  return h;
}

struct RayTracer {
  PacketLds<64>& lds;
  bool store;
  __device__ Hit operator()(const SceneView& s, D3 o, D3 d, double tmax) { return trace_rays(s, o, d, tmax, lds); }
  __device__ bool stores() const { return store; }
};

// ------------------------------------------------ 4 x 4 rays, four lanes each

// The value of the lane whose number in its quad differs by kXor (1 or 2).
template <int kXor>
__device__ __forceinline__ int quad_swap(int v) {
  constexpr int kCtrl = kXor == 1 ? 0xB1 : 0x4E;  // quad_perm [1,0,3,2], [2,3,0,1]
  return __builtin_amdgcn_update_dpp(0, v, kCtrl, 0xF, 0xF, false);
}
template <int kXor>
__device__ __forceinline__ double quad_swap(double v) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)quad_swap<kXor>((int)(unsigned)u);
  const unsigned hi = (unsigned)quad_swap<kXor>((int)(unsigned)(u >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
template <int kXor>
__device__ __forceinline__ void quad_nearest(Hit& h) {
  const double t = quad_swap<kXor>(h.t);
  const int tri = quad_swap<kXor>(h.tri);
  if (tri >= 0 && hit_before(t, tri, h)) h = Hit{t, tri};
}

// Bit q set: some ray's lane q has its bit of b set.
__device__ __forceinline__ uint32_t any_of_quads(unsigned long long b) {
  uint32_t m = (uint32_t)(b | b >> 32);
  m |= m >> 16;
  m |= m >> 8;
  m |= m >> 4;
  return m & 15u;
}

__device__ Hit trace_quads(const SceneView& s, D3 o, D3 d, double tmax, PacketLds<16>& lds) {
  const int lane = threadIdx.x, q = lane & 3, slot = lane >> 2;
  Hit h{tmax, -1};  // the same in a quad's lanes
  BoxRay r = packet_box_ray(s, o, d, tmax);
  const int oct = packet_octant(d);
  const int pair = oct < 4 ? oct : oct ^ 7;
  int sp = 0;
  uint32_t cur = 0;
  while (true) {
    const int count = (int)(cur & 7u);
    const uint32_t first = cur >> 3;
    if (count == 0) {
      const float4* c = reinterpret_cast<const float4*>(s.nodes + first);
      const float4 a0 = c[2 * q], a1 = c[2 * q + 1], b0 = c[2 * q + 8], b1 = c[2 * q + 9];
      const uint32_t* words = reinterpret_cast<const uint32_t*>(s.nodes + first);
      uint32_t after0 = words[16 * pair + 7] >> (8 * q) & 0xFFu, after1 = words[16 * pair + 15] >> (8 * q) & 0xFFu;
      float near0, near1;
      const bool hit0 = box_test(r, a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, near0);
      const bool hit1 = box_test(r, b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, near1);
      const uint32_t hits = any_of_quads(__ballot(hit0)) | any_of_quads(__ballot(hit1)) << 4;
      if (oct >= 4) {
        after0 = ~(after0 | 1u << q);
        after1 = ~(after1 | 16u << q);
      }
      after0 &= hits;
      after1 &= hits;
      const bool any0 = hits >> q & 1u, any1 = hits >> q & 16u;
      const bool top0 = any0 && after0 == (hits ^ 1u << q), top1 = any1 && after1 == (hits ^ 16u << q);
      const uint32_t ref0 = __float_as_uint(a1.z), ref1 = __float_as_uint(b1.z);
      // positions below kTraceStack (the build's bound)
      const int pos0 = sp + __builtin_popcount(after0), pos1 = sp + __builtin_popcount(after1);
      if (any0 && !top0) {
        if (pos0 < kNearStack) lds.near[pos0 * 16 + slot] = hit0 ? near0 : __builtin_inff();
        if (slot == 0) lds.ref[pos0] = ref0;
      }
      if (any1 && !top1) {
        if (pos1 < kNearStack) lds.near[pos1 * 16 + slot] = hit1 ? near1 : __builtin_inff();
        if (slot == 0) lds.ref[pos1] = ref1;
      }
      if (hits != 0u) {  // the nearest child is visited next, without a turn through the stack
        cur = (uint32_t)__builtin_amdgcn_readlane((int)(top0 ? ref0 : ref1), __builtin_ctzll(__ballot(top0 || top1)));
        sp += __builtin_popcount(hits) - 1;
        continue;
      }
    } else {
      const TriGeo g = s.geo[first + q];  // padded: in bounds for every leaf
      const TriTerms k = tri_terms(g, o, d);
      const bool maybe = q < count && tri_maybe(k, h.t);
      if (any_lane(maybe)) {
        double th;
        if (maybe && tri_accept(k, h.t, &th) && hit_before(th, (int)first + q, h)) h = Hit{th, (int)first + q};
        quad_nearest<1>(h);
        quad_nearest<2>(h);
        if (h.tri >= 0) r.tmax = box_tmax(h.t, r.entry);
      }
    }
    if (!packet_pop(lds, slot, r.tmax, sp, cur)) break;
  }
  if (h.tri >= 0) h.tri = s.order[h.tri];
  return h;
}

struct QuadTracer {
  PacketLds<16>& lds;
  bool store;
  __device__ Hit operator()(const SceneView& s, D3 o, D3 d, double tmax) { return trace_quads(s, o, d, tmax, lds); }
  __device__ bool stores() const { return store; }
};

template <class Tracer>
__device__ __forceinline__ void shade(Tracer& tr, const SceneView& s, const RayCam& rc, int x, int y, int w, int h,
                                      int mode, float* a, float* b, float* c) {
  if (mode == 1)
    shade_rsm(tr, s, rc, x, y, w, h, a, b, c);  // diffuse, normal, depth
  else if (mode == 2)
    shade_surface(tr, s, rc, x, y, w, h, a, b);  // albedo, VSM moments
  else
    shade_gbuffer(tr, s, rc, x, y, w, h, a, b);  // depth, normal
}

// Lanes past the image repeat its last row or column (the whole wave runs the
// packet) and store nothing.
__global__ __launch_bounds__(64) void raycast_kernel(SceneView s, RayCam rc, int w, int h, int mode,
                                                      float* __restrict__ a, float* __restrict__ b,
                                                      float* __restrict__ c) {
  __shared__ PacketLds<64> lds;
  const int x = blockIdx.x * 8 + (threadIdx.x & 7);
  const int y = blockIdx.y * 8 + (threadIdx.x >> 3);
  RayTracer tr{lds, x < w && y < h};
  shade(tr, s, rc, min(x, w - 1), min(y, h - 1), w, h, mode, a, b, c);
}

__global__ __launch_bounds__(64) void raycast_quad_kernel(SceneView s, RayCam rc, int w, int h, int mode,
                                                           float* __restrict__ a, float* __restrict__ b,
                                                           float* __restrict__ c) {
  __shared__ PacketLds<16> lds;
  const int q = threadIdx.x & 3, r = threadIdx.x >> 2;
  const int x = blockIdx.x * 4 + (r & 3);
  const int y = blockIdx.y * 4 + (r >> 2);
  QuadTracer tr{lds, q == 0 && x < w && y < h};
  shade(tr, s, rc, min(x, w - 1), min(y, h - 1), w, h, mode, a, b, c);
}

struct RsmJobs {
  RsmJob j[kRsmJobs];
};
static_assert(sizeof(RsmJobs) + 2 * sizeof(int) <= 4096, "kernel arguments");

// The RSM of job blockIdx.z, as the two kernels above.
__global__ __launch_bounds__(64) void rsms_kernel(RsmJobs jobs, int w, int h) {
  __shared__ PacketLds<64> lds;
  const RsmJob& job = jobs.j[blockIdx.z];
  const int x = blockIdx.x * 8 + (threadIdx.x & 7);
  const int y = blockIdx.y * 8 + (threadIdx.x >> 3);
  RayTracer tr{lds, x < w && y < h};
  shade_rsm(tr, job.scene, job.light, min(x, w - 1), min(y, h - 1), w, h, job.diffuse, job.normal, job.depth);
}
__global__ __launch_bounds__(64) void rsms_quad_kernel(RsmJobs jobs, int w, int h) {
  __shared__ PacketLds<16> lds;
  const RsmJob& job = jobs.j[blockIdx.z];
  const int q = threadIdx.x & 3, r = threadIdx.x >> 2;
  const int x = blockIdx.x * 4 + (r & 3);
  const int y = blockIdx.y * 4 + (r >> 2);
  QuadTracer tr{lds, q == 0 && x < w && y < h};
  shade_rsm(tr, job.scene, job.light, min(x, w - 1), min(y, h - 1), w, h, job.diffuse, job.normal, job.depth);
}

}  // namespace

hipError_t launch_rsms(hipStream_t st, const RsmJob* jobs, int n, int w, int h) {
  for (int i = 0; i < n; i += kRsmJobs) {
    const int m = n - i < kRsmJobs ? n - i : kRsmJobs;
    RsmJobs group = {};
    for (int k = 0; k < m; ++k) group.j[k] = jobs[i + k];
    if ((size_t)w * (size_t)h * (size_t)m <= kWideRays)
      hipLaunchKernelGGL(rsms_quad_kernel, dim3((w + 3) / 4, (h + 3) / 4, m), dim3(64), 0, st, group, w, h);
    else
      hipLaunchKernelGGL(rsms_kernel, dim3((w + 7) / 8, (h + 7) / 8, m), dim3(64), 0, st, group, w, h);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_raycast(hipStream_t st, const SceneView& s, const RayCam& rc, int w, int h, int rsm,
                          float* a, float* b, float* c) {
  if ((size_t)w * (size_t)h <= kWideRays) {
    const dim3 grid((w + 3) / 4, (h + 3) / 4);
    hipLaunchKernelGGL(raycast_quad_kernel, grid, dim3(64), 0, st, s, rc, w, h, rsm, a, b, c);
  } else {
    const dim3 grid((w + 7) / 8, (h + 7) / 8);
    hipLaunchKernelGGL(raycast_kernel, grid, dim3(64), 0, st, s, rc, w, h, rsm, a, b, c);
  }
  return hipGetLastError();
}

}  // namespace mlgi
