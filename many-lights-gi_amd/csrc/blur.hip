// Geometry-aware separable blur of the irradiance: gi/gi_blur.frag:24-72 as
// GIStage::blur runs it (GIStage.cpp:308-344), an x pass into a temporary and
// a y pass of the temporary, both weighted by the face normals and the
// linear depth (reprojection.glsl:6-13). Compiled with -ffp-contract=off and
// written in the oracle's operation order, so the result is bit-exact
// against its FP32 instantiation.
//
// Both passes are fused: a workgroup owns a kTw x kTh output tile, loads the
// irradiance, decoded normals and linear depths of the tile plus a 3-texel
// apron into LDS once, runs the x pass over the kTh + 6 rows the y pass needs
// (into LDS) and then the y pass. HBM traffic per pixel: the 28 input bytes
// (plus the apron, mostly served by L2) and the 12 output bytes, against two
// full-screen read/write passes in the reference. Out-of-range texels read 0
// (irradiance 0, normal (-1, -1, -1), depth 0), as the x pass's temporary does
// outside the image.
//
// Bound: VALU issue (77% of it with 32 x 8 tiles and one pixel per lane, 667
// instructions per wave of pixels, 43.8 us at 1080p). So a lane blurs kRun
// neighbouring pixels of a line: the samples they share are read once (two
// 16-byte LDS reads each), a weight is the same for both ends of a pair, bit
// for bit (its dot product's factors and its depth difference only trade
// places), and is formed once for the pairs within a run, the three channels'
// quotients share one reciprocal, a taller tile's apron costs fewer extra rows
// (1.375 per row at 16, 1.75 at 8), and all loads of a tile are in flight at
// once: 25.1 us at 1080p, and down to 130 x 109 no slower than the smaller
// forms. Other forms at 1080p: 32 x 16 tiles with one pixel per lane 27.9,
// with two 28.1, with four 38.5 (a third of the waves); 32 x 8 with one 32.9.
#include "kernels.hpp"
#include "mlgi_device.hpp"

namespace mlgi {
namespace {

constexpr int kRadius = 3;
constexpr int kTw = 64, kTh = 16, kRun = 2;
constexpr int kThreads = kTw * kTh / kRun;                       // one run of the y pass per lane
constexpr int kAw = kTw + 2 * kRadius, kAh = kTh + 2 * kRadius;  // apron region
constexpr int kPitch = kAw + 1;                                  // LDS row pitch in texels (bank spread)
constexpr int kLine = kRun + 2 * kRadius;                        // the samples of a run

// a / b for b in [1, 7] from y = RN(1 / b): dev::div_rn's IEEE quotient (below
// 2^-120 it may be off by its last bit), an infinite a kept.
__device__ __forceinline__ float by_weight(float a, float b, float y) {
  const float q = dev::div_rn(a, b, y);
  return fabsf(a) == __builtin_inff() ? a : q;
}

// -B / (A + zn) (dev::div_rn; where the division gives an infinity this gives
// NaN, and a weight is 0 either way).
__device__ __forceinline__ float linear_depth(float d, float A, float B) {
  const float zn = 2.0f * d - 1.0f;
  const float w = A + zn;
  return dev::div_rn(-B, w, dev::recip_rn(w));
}

// The weight of gi_blur.frag's processSample between two texels k apart
// (normal in xyz, linear depth in w).
__device__ __forceinline__ float pair_factor(const float4& c, const float4& s, int k) {
  const float nf = 1.0f - fmaxf(c.x * s.x + c.y * s.y + c.z * s.z, 0.0f);
  const float dd = s.w - c.w;
  const float nd = nf * 5.0f;
  return fmaxf(((float)kRadius - (float)k + 1.0f) / 4.0f - dd * dd - nd * nd, 0.0f);
}

// Blurs the kRun middle ones of kLine consecutive texels: geometry n, values
// g, results r (rgb).
__device__ __forceinline__ void blur_line(const float4 (&n)[kLine], const float4 (&g)[kLine], float (&r)[kRun][3]) {
  float f[kLine][kRadius + 1];  // f[a][k]: the weight of texels a and a + k
#pragma unroll
  for (int a = 0; a < kLine; ++a)
#pragma unroll
    for (int k = 1; k <= kRadius; ++k) {
      const int b = a + k;
      const bool used = (a >= kRadius && a < kRadius + kRun) || (b >= kRadius && b < kRadius + kRun);
      f[a][k] = used && b < kLine ? pair_factor(n[a], n[b], k) : 0.0f;
    }
#pragma unroll
  for (int o = 0; o < kRun; ++o) {
    const int c = o + kRadius;
    float ar = g[c].x, ag = g[c].y, ab = g[c].z, fsum = 1.0f;
#pragma unroll
    for (int side = -1; side <= 1; side += 2)
#pragma unroll
      for (int k = 1; k <= kRadius; ++k) {
        const int s = c + side * k;
        const float w = side < 0 ? f[s][k] : f[c][k];
        fsum = fsum + w;
        ar = ar + g[s].x * w;
        ag = ag + g[s].y * w;
        ab = ab + g[s].z * w;
      }
    const float y = dev::recip_rn(fsum);
    r[o][0] = by_weight(ar, fsum, y);
    r[o][1] = by_weight(ag, fsum, y);
    r[o][2] = by_weight(ab, fsum, y);
  }
}

__global__ __launch_bounds__(kThreads) void gi_blur_kernel(const float* __restrict__ gi,
                                                           const float* __restrict__ normal,
                                                           const float* __restrict__ depth, int w, int h, float A,
                                                           float B, float* __restrict__ out) {
  __shared__ float4 sn[kAh * kPitch];  // decoded normal, linear depth
  __shared__ float4 sg[kAh * kPitch];  // irradiance, then the x pass's result (columns 0 .. kTw - 1)
  const int tid = threadIdx.x;
  const int x0 = blockIdx.x * kTw, y0 = blockIdx.y * kTh;

  // every load of the tile is requested before the first is used
  constexpr int kTexels = kAw * kAh, kLoads = (kTexels + kThreads - 1) / kThreads;
  float v[kLoads][7];
  bool in[kLoads];
#pragma unroll
  for (int t = 0; t < kLoads; ++t) {
    const int i = tid + t * kThreads;
    const int ly = i / kAw, lx = i % kAw;
    const int x = x0 + lx - kRadius, y = y0 + ly - kRadius;
    in[t] = x >= 0 && y >= 0 && x < w && y < h && i < kTexels;
    const size_t q = in[t] ? (size_t)y * w + x : 0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      v[t][k] = gi[q * 3 + k];
      v[t][3 + k] = normal[q * 3 + k];
    }
    v[t][6] = depth[q];
  }
#pragma unroll
  for (int t = 0; t < kLoads; ++t) {
    const int i = tid + t * kThreads;
    if (i >= kTexels) continue;
#pragma unroll
    for (int k = 0; k < 7; ++k) v[t][k] = in[t] ? v[t][k] : 0.0f;
    const int at = (i / kAw) * kPitch + i % kAw;
    sg[at] = make_float4(v[t][0], v[t][1], v[t][2], 0.0f);
    sn[at] = make_float4(v[t][3] * 2.0f - 1.0f, v[t][4] * 2.0f - 1.0f, v[t][5] * 2.0f - 1.0f,
                         linear_depth(v[t][6], A, B));
  }
  __syncthreads();

  // x pass over every apron row (rows outside the image stay 0): runs of kRun
  // columns, neighbouring lanes on neighbouring rows
  constexpr int kXRuns = kAh * (kTw / kRun), kXTurns = (kXRuns + kThreads - 1) / kThreads;
  float xr[kXTurns][kRun][3];
#pragma unroll
  for (int t = 0; t < kXTurns; ++t) {
    const int i = tid + t * kThreads;
    if (i < kXRuns) {
      const int at = (i % kAh) * kPitch + (i / kAh) * kRun;
      float4 n[kLine], g[kLine];
#pragma unroll
      for (int k = 0; k < kLine; ++k) {
        n[k] = sn[at + k];
        g[k] = sg[at + k];
      }
      blur_line(n, g, xr[t]);
    }
  }
  __syncthreads();  // the irradiance is read: its place takes the results
#pragma unroll
  for (int t = 0; t < kXTurns; ++t) {
    const int i = tid + t * kThreads;
    if (i < kXRuns) {
      const int ly = i % kAh, y = y0 + ly - kRadius;
      const bool row = y >= 0 && y < h;
#pragma unroll
      for (int o = 0; o < kRun; ++o)
        sg[ly * kPitch + (i / kAh) * kRun + o] =
            make_float4(row ? xr[t][o][0] : 0.0f, row ? xr[t][o][1] : 0.0f, row ? xr[t][o][2] : 0.0f, 0.0f);
    }
  }
  __syncthreads();

  // y pass of the tile's pixels: runs of kRun rows
  {
    const int tx = tid % kTw, ty = (tid / kTw) * kRun;
    const int x = x0 + tx;
    float4 n[kLine], g[kLine];
#pragma unroll
    for (int k = 0; k < kLine; ++k) {
      n[k] = sn[(ty + k) * kPitch + tx + kRadius];
      g[k] = sg[(ty + k) * kPitch + tx];
    }
    float r[kRun][3];
    blur_line(n, g, r);
#pragma unroll
    for (int o = 0; o < kRun; ++o) {
      const int y = y0 + ty + o;
      if (x < w && y < h) {
        float* p = out + ((size_t)y * w + x) * 3;
        // a stream past the L2s: 25.6 -> 25.1 us at 1080p; with the composite
        // that reads it, plain / streamed: 640 x 360 11.7/12.3, 1080p 53.0/54.3, 4K 203/199
        __builtin_nontemporal_store(r[o][0], p);
        __builtin_nontemporal_store(r[o][1], p + 1);
        __builtin_nontemporal_store(r[o][2], p + 2);
      }
    }
  }
}

}  // namespace

hipError_t launch_gi_blur(hipStream_t s, const float* gi, const float* normal, const float* depth, int w, int h,
                          const float* projection16, float* out) {
  const dim3 grid((w + kTw - 1) / kTw, (h + kTh - 1) / kTh);
  hipLaunchKernelGGL(gi_blur_kernel, grid, dim3(kThreads), 0, s, gi, normal, depth, w, h, projection16[10],
                     projection16[14], out);
  return hipGetLastError();
}

}  // namespace mlgi
