// Device point generation: the area-proportional point set of a scene
// (what the reference's tessellation and geometry shaders emit per frame,
// ism.tesc:11-23, ism.geom:49-69) sampled on the GPU and grouped by bin,
// for scenes whose point sets are built at run time. Each lane samples one
// point with the host sampler's double-precision code (scene_trace.hpp,
// compiled with -ffp-contract=off in both), so record i and its bin equal
// the host's; bins are counted with atomics, whose returned counts are the
// points' places in their bins, and scanned by one workgroup. Within a bin the
// records come in no fixed order: every consumer (the splat) takes a minimum
// over the bin's splats, which no order changes.
//
// Atomics in memory run at about 12 G/s over the chip's eight L2s, less on few
// counters, and bound the sampling at one per point. Each workgroup therefore
// counts a run of points of its own in LDS, and the counts of all workgroups
// are scanned per bin (1M points in 4,096 bins: 87 us of sampling and 15 of
// moving the records -> 35, 18 and 6 of scanning). What is left is the search
// for the triangle and its vertices, 64 different lines a wave and step: the
// search starts in LDS (45 -> 35 us).
//
// The table of counts costs as much as the atomics where a bin has few points
// or the bins are many; there each point keeps its atomic in memory. The whole
// call, memory / LDS, in us:
//   1M points in 256 / 1,024 / 4,096 / 8,192 bins: 523/96, 267/100, 143/107, 122/119
//   4M points in 4,096 / 8,192 bins: 661/610, 582/631
//   64 points a bin, 256 / 1,024 / 4,096 bins: 34/29, 39/31, 88/76
//   24 points a bin, 4,096 bins: 57/70
#include "kernels.hpp"
#include "scene_trace.hpp"

namespace mlgi {
namespace {

using namespace mlgi_scene_impl;

// Workgroups that count in LDS (two per CU at most), the bins they count and
// the points per bin from which they do.
constexpr int kHistGroups = 512, kHistBins = 4096, kHistPoints = 64;
// Running areas kept in LDS for the first steps of the search (16 KB).
constexpr int kEnds = 2048;

__global__ __launch_bounds__(256) void fill_u32_kernel(uint32_t* __restrict__ p, int n, uint32_t v) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) p[i] = v;
}

__global__ __launch_bounds__(256) void point_sample_kernel(const Tri* __restrict__ tris,
                                                           const double* __restrict__ cdf, int nt, double total,
                                                           uint64_t seed, float r_packed, int n_bins, int n,
                                                           float4* __restrict__ tmp, uint2* __restrict__ place,
                                                           uint32_t* __restrict__ count) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float rec[4];
  int b;
  sample_point(tris, cdf, nt, total, seed, (uint64_t)i, r_packed, n_bins, rec, &b);
  tmp[i] = make_float4(rec[0], rec[1], rec[2], rec[3]);
  place[i] = make_uint2((uint32_t)b,
                        __hip_atomic_fetch_add(&count[b], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// The same with the places counted in LDS: workgroup g samples the points
// [g * chunk, g * chunk + chunk) and writes its counts as row g of hist. 16
// waves and 32 KB of LDS a workgroup.
__global__ __launch_bounds__(1024) void point_sample_hist_kernel(const Tri* __restrict__ tris,
                                                                 const double* __restrict__ cdf, int nt, double total,
                                                                 uint64_t seed, float r_packed, int n_bins, int n,
                                                                 int chunk, float4* __restrict__ tmp,
                                                                 uint2* __restrict__ place,
                                                                 uint32_t* __restrict__ hist) {
  __shared__ uint32_t cnt[kHistBins];
  // running areas at the ends of runs of `step` triangles
  __shared__ double ends[kEnds];
  const int step = (nt + kEnds - 1) / kEnds, n_ends = (nt + step - 1) / step;
  for (int k = threadIdx.x; k < n_ends; k += 1024) ends[k] = cdf[min(nt, (k + 1) * step) - 1];
  for (int b = threadIdx.x; b < n_bins; b += 1024) cnt[b] = 0;
  __syncthreads();
  const int64_t i0 = (int64_t)blockIdx.x * chunk, i1 = i0 + chunk < n ? i0 + chunk : n;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += 1024) {
    const double u = point_area(total, seed, (uint64_t)i);
    const int t0 = upper_bound_d(ends, n_ends, u) * step;
    const int ti = t0 < nt ? t0 + upper_bound_d(cdf + t0, min(step, nt - t0), u) : nt;
    float rec[4];
    int b;
    sample_on(tris, ti, nt, seed, (uint64_t)i, r_packed, n_bins, rec, &b);
    tmp[i] = make_float4(rec[0], rec[1], rec[2], rec[3]);
    place[i] = make_uint2((uint32_t)b, atomicAdd(&cnt[b], 1u));
  }
  __syncthreads();
  for (int b = threadIdx.x; b < n_bins; b += 1024) hist[(size_t)blockIdx.x * n_bins + b] = cnt[b];
}

// Per bin: exclusive scan of hist's rows in place, total into count. A
// workgroup takes 64 bins, each of its waves kHistGroups / 16 rows, whose
// loads are in flight together.
__global__ __launch_bounds__(1024) void hist_scan_kernel(uint32_t* __restrict__ hist, int rows, int n_bins,
                                                         uint32_t* __restrict__ count) {
  constexpr int kPer = kHistGroups / 16;
  __shared__ uint32_t part[16][64];
  const int lane = threadIdx.x & 63, seg = threadIdx.x >> 6, b = blockIdx.x * 64 + lane;
  uint32_t v[kPer], s = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int g = seg * kPer + k;
    v[k] = g < rows && b < n_bins ? hist[(size_t)g * n_bins + b] : 0u;
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) s += v[k];
  part[seg][lane] = s;
  __syncthreads();
  uint32_t run = 0;
  for (int k = 0; k < seg; ++k) run += part[k][lane];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int g = seg * kPer + k;
    if (g < rows && b < n_bins) hist[(size_t)g * n_bins + b] = run;
    run += v[k];
  }
  if (seg == 15 && b < n_bins) count[b] = run;
}

// Exclusive scan of count[0, n_bins) into offsets[0, n_bins] (one workgroup
// of 1024 lanes, each owning a contiguous run of bins).
__global__ __launch_bounds__(1024) void bin_scan_kernel(const uint32_t* __restrict__ count, int n_bins,
                                                        uint32_t* __restrict__ offsets) {
  __shared__ uint32_t part[1024];
  const int t = threadIdx.x;
  const int per = (n_bins + 1023) / 1024;
  const int b0 = min(n_bins, t * per), b1 = min(n_bins, b0 + per);
  uint32_t s = 0;
  for (int b = b0; b < b1; ++b) s += count[b];
  part[t] = s;
  __syncthreads();
  // inclusive Hillis-Steele scan of the 1024 run sums
  for (int o = 1; o < 1024; o <<= 1) {
    const uint32_t v = t >= o ? part[t - o] : 0u;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  uint32_t run = t > 0 ? part[t - 1] : 0u;
  for (int b = b0; b < b1; ++b) {
    offsets[b] = run;
    run += count[b];
  }
  if (t == 1023) offsets[n_bins] = part[1023];
}

__global__ __launch_bounds__(256) void point_scatter_kernel(const float4* __restrict__ tmp,
                                                            const uint2* __restrict__ place, int n,
                                                            const uint32_t* __restrict__ offsets,
                                                            float4* __restrict__ records) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint2 p = place[i];
  records[offsets[p.x] + p.y] = tmp[i];
}

// The same for places in a workgroup's run: on the grid of the sampling, so
// that a row of hist is read by one workgroup, on the XCD that wrote its points
// (17.7 us for 1M points; a lane per point on a grid of its own: 22.4).
__global__ __launch_bounds__(1024) void point_scatter_hist_kernel(const float4* __restrict__ tmp,
                                                                  const uint2* __restrict__ place, int n,
                                                                  const uint32_t* __restrict__ offsets,
                                                                  const uint32_t* __restrict__ hist, int chunk,
                                                                  int n_bins, float4* __restrict__ records) {
  const uint32_t* row = hist + (size_t)blockIdx.x * n_bins;
  const int64_t i0 = (int64_t)blockIdx.x * chunk, i1 = i0 + chunk < n ? i0 + chunk : n;
  for (int64_t i = i0 + threadIdx.x; i < i1; i += 1024) {
    const uint2 p = place[i];
    records[offsets[p.x] + row[p.x] + p.y] = tmp[i];
  }
}

unsigned blocks_for(int n) { return (unsigned)((n + 255) / 256); }

}  // namespace

int points_hist_rows(int n, int n_bins) {
  if (n_bins > kHistBins || n < (int64_t)kHistPoints * n_bins) return 0;
  const int rows = (int)(((int64_t)n + 1023) / 1024);
  return rows < kHistGroups ? rows : kHistGroups;
}

hipError_t launch_sample_points(hipStream_t s, const Tri* tris, const double* cdf, int nt, double total,
                                uint64_t seed, float r_packed, int n_bins, int n, float* tmp, uint2* place,
                                uint32_t* count, uint32_t* hist, float* records, uint32_t* offsets) {
  hipError_t e;
  const int rows = hist ? points_hist_rows(n, n_bins) : 0;
  const int chunk = rows ? (int)(((int64_t)n + rows - 1) / rows) : 1;
  if (rows) {
    hipLaunchKernelGGL(point_sample_hist_kernel, dim3(rows), dim3(1024), 0, s, tris, cdf, nt,
                       total, seed, r_packed, n_bins, n, chunk, reinterpret_cast<float4*>(tmp), place, hist);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(hist_scan_kernel, dim3((n_bins + 63) / 64), dim3(1024), 0, s, hist, rows, n_bins, count);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(bin_scan_kernel, dim3(1), dim3(1024), 0, s, count, n_bins, offsets);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(point_scatter_hist_kernel, dim3(rows), dim3(1024), 0, s, reinterpret_cast<const float4*>(tmp),
                       place, n, offsets, hist, chunk, n_bins, reinterpret_cast<float4*>(records));
    return hipGetLastError();
  }
  hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks_for(n_bins) < 1024 ? blocks_for(n_bins) : 1024), dim3(256), 0, s,
                     count, n_bins, 0u);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (n > 0) {
    hipLaunchKernelGGL(point_sample_kernel, dim3(blocks_for(n)), dim3(256), 0, s, tris, cdf, nt, total, seed, r_packed,
                       n_bins, n, reinterpret_cast<float4*>(tmp), place, count);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  hipLaunchKernelGGL(bin_scan_kernel, dim3(1), dim3(1024), 0, s, count, n_bins, offsets);
  if ((e = hipGetLastError()) != hipSuccess || n == 0) return e;
  hipLaunchKernelGGL(point_scatter_kernel, dim3(blocks_for(n)), dim3(256), 0, s, reinterpret_cast<const float4*>(tmp),
                     place, n, offsets, reinterpret_cast<float4*>(records));
  return hipGetLastError();
}

}  // namespace mlgi
