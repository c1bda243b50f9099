// Deferred composite: direct light with a VSM shadow, GI ambient, Reinhard
// tone mapping and gamma 2.2 (deferredshading.frag:47-81 with
// shadowmapping.glsl:6-34 and srgb_utils.glsl, bound by
// DeferredShadingStage::process, DeferredShadingStage.cpp:76-131), one lane
// per pixel over 64 x 4 tiles (a wave's row of three-float texels is 768
// contiguous bytes). 44 bytes are read (depth, normal, diffuse, specular, GI,
// occlusion) and 12 written per pixel, plus four bilinear taps of the VSM
// moments.
//
// Bound: with the library's powf (ten per pixel) and IEEE division sequences
// (17) it was VALU issue, 82 us for 1080p. The quotients are formed from the
// correctly rounded reciprocals of their divisors (dev::div_rn: the same bits;
// operands outside its range take the division), the three divisions by one
// length or w share one reciprocal, and the powers of the gamma are formed
// from the hardware's base-2 logarithm and exponential (pow_pos): 36.9 us.
//
// Conventions (the oracle's): the pixel is sampled at its centre; the world
// position is inverse(P*V) of the centre's NDC; the VSM is sampled
// bilinearly with a (0, 0) border; pow(0, y) = 0; a null specular buffer
// reads 0 and a null occlusion buffer reads 1. FP32 throughout.
#include "kernels.hpp"
#include "mlgi_device.hpp"

namespace mlgi {
namespace {

__device__ __forceinline__ float clamp01(float x) { return fminf(fmaxf(x, 0.0f), 1.0f); }

// a, b, c divided by d: dev::div_rn's IEEE quotients from one reciprocal where
// d is a plain number, the division where it is zero, tiny, huge or not
// finite, or a numerator is huge.
__device__ __forceinline__ void divide(float& a, float& b, float& c, float d) {
  const float m = fabsf(d), n = fmaxf(fmaxf(fabsf(a), fabsf(b)), fabsf(c));
  if (m >= 0x1p-40f && m <= 0x1p40f && n <= 0x1p60f) {
    const float y = dev::recip_rn(d);
    a = dev::div_rn(a, d, y);
    b = dev::div_rn(b, d, y);
    c = dev::div_rn(c, d, y);
  } else {
    a = a / d, b = b / d, c = c / d;
  }
}
// a / b for plain numbers.
__device__ __forceinline__ float quotient(float a, float b) { return dev::div_rn(a, b, dev::recip_rn(b)); }
// a / b for any: an infinite moment or colour, a window or sum that is 0 or
// huge take the division, whose infinities the clamps turn into 0 or 1.
__device__ __forceinline__ float quotient_any(float a, float b) {
  const float m = fabsf(b);
  return m >= 0x1p-40f && m <= 0x1p40f && fabsf(a) <= 0x1p60f ? quotient(a, b) : a / b;
}

__device__ __forceinline__ float smoothstep_f(float e0, float e1, float x) {
  const float t = clamp01(quotient_any(x - e0, e1 - e0));
  return t * t * (3.0f - 2.0f * t);
}

// x^y for x > 0 (0 otherwise), y = 2.2 or 1 / 2.2: 2^(y log2 x) with x = m 2^e,
// m in [0.75, 1.5), so that the hardware logarithm's error is one of a value
// below 0.6, and y e split from the sum with its rounding error before the
// exponential takes the fraction; ~20 instructions. Over all significands at 12
// exponents the gamma is off by at most 1.03 ulp, 0.26 on average (the library's
// powf here: 1.32 and 0.34). The same in FP64, 0.503 ulp, takes 49 us in place
// of 37 at 1080p.
__device__ __forceinline__ float pow_pos(float x, float y) {
  const float h = __builtin_amdgcn_frexp_mantf(x);  // [0.5, 1)
  const bool low = h < 0.75f;
  const float m = low ? h + h : h;
  const float e = (float)(__builtin_amdgcn_frexp_expf(x) - (low ? 1 : 0));
  const float l = __builtin_amdgcn_logf(m);
  const float p = y * e;
  const float n = rintf(__builtin_fmaf(y, l, p));
  const float f = (p - n) + __builtin_fmaf(y, l, __builtin_fmaf(y, e, -p));
  const float r = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
  return x > 0.0f ? r : 0.0f;
}

// x^20 for x >= 0: products in FP64 round once (0.51 ulp). Seen through the
// gamma, in units of 2^-23: 0.94 at most; five products in FP32 3.76, powf 1.39.
__device__ __forceinline__ float pow20(float x) {
  const double x1 = (double)x, x2 = x1 * x1, x4 = x2 * x2, x5 = x4 * x1, x10 = x5 * x5;
  return (float)(x10 * x10);
}

// shadowmapping.glsl:13-20
__device__ __forceinline__ float vsm_factor(float mx, float my, float compare) {
  const float p = smoothstep_f(compare - 0.001f, compare, mx);
  // E[d^2] - E[d]^2 cancels: one rounding (fused) instead of two
  const float variance = fmaxf(__builtin_fmaf(-mx, mx, my), 0.001f);
  const float d = compare - mx;
  const float p_max = clamp01(quotient(quotient_any(variance, variance + d * d) - 0.1f, 1.0f - 0.1f));
  return clamp01(fmaxf(p, p_max));
}

__global__ __launch_bounds__(256) void composite_kernel(CompositeArgs a) {
  const int x = blockIdx.x * 64 + (threadIdx.x & 63);
  const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (x >= a.w || y >= a.h) return;
  const size_t c = (size_t)y * a.w + x;
  const float u = quotient((float)x + 0.5f, (float)a.w), v = quotient((float)y + 0.5f, (float)a.h);
  const float ndc[4] = {u * 2.0f - 1.0f, v * 2.0f - 1.0f, a.depth[c] * 2.0f - 1.0f, 1.0f};
  float r[4];
#pragma unroll
  for (int row = 0; row < 4; ++row) {
    float acc = 0.0f;
#pragma unroll
    for (int col = 0; col < 4; ++col) acc += a.vp_inv[col * 4 + row] * ndc[col];
    r[row] = acc;
  }
  float wx = r[0], wy = r[1], wz = r[2];
  divide(wx, wy, wz, r[3]);
  const float nx = a.normal[c * 3] * 2.0f - 1.0f, ny = a.normal[c * 3 + 1] * 2.0f - 1.0f,
              nz = a.normal[c * 3 + 2] * 2.0f - 1.0f;
  const float lx = a.inv_light_dir[0], ly = a.inv_light_dir[1], lz = a.inv_light_dir[2];
  float vx = a.eye[0] - wx, vy = a.eye[1] - wy, vz = a.eye[2] - wz;
  const float vl = sqrtf(vx * vx + vy * vy + vz * vz);
  divide(vx, vy, vz, vl);
  float hx = lx + vx, hy = ly + vy, hz = lz + vz;
  const float hl = sqrtf(hx * hx + hy * hy + hz * hz);
  divide(hx, hy, hz, hl);
  const float ndotl = nx * lx + ny * ly + nz * lz;
  const float ndoth = nx * hx + ny * hy + nz * hz;
  float sc[4];
  const float wp[4] = {wx, wy, wz, 1.0f};
#pragma unroll
  for (int row = 0; row < 4; ++row) {
    float acc = 0.0f;
#pragma unroll
    for (int col = 0; col < 4; ++col) acc += a.blvp[col * 4 + row] * wp[col];
    sc[row] = acc;
  }
  // bilinear VSM moments, border (0, 0)
  float cx = sc[0], cy = sc[1], cz = 0.0f;
  divide(cx, cy, cz, sc[3]);
  const float s = cx * (float)a.vw - 0.5f, t = cy * (float)a.vh - 0.5f;
  const float fs = floorf(s), ft = floorf(t);
  const float fa = s - fs, fb = t - ft;
  float mx = 0.0f, my = 0.0f;
  if (fabsf(fs) < 1e9f && fabsf(ft) < 1e9f) {  // far outside: all border
    const int i0 = (int)fs, j0 = (int)ft;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = i0 + (k & 1), j = j0 + (k >> 1);
      const float wgt = ((k & 1) ? fa : 1.0f - fa) * ((k >> 1) ? fb : 1.0f - fb);
      const bool in = i >= 0 && j >= 0 && i < a.vw && j < a.vh;
      const float2 m = reinterpret_cast<const float2*>(a.vsm)[in ? (size_t)j * a.vw + i : 0];
      mx += in ? wgt * m.x : 0.0f;
      my += in ? wgt * m.y : 0.0f;
    }
  }
  const float dlx = wx - a.light_pos[0], dly = wy - a.light_pos[1], dlz = wz - a.light_pos[2];
  const float dist = sqrtf(dlx * dlx + dly * dly + dlz * dlz);
  const float shadow = vsm_factor(mx, my, dist) * (sc[3] > 0.0f ? 1.0f : 0.0f);
  const float occ = a.occlusion ? a.occlusion[c] : 1.0f;
  const float spec_f = pow20(fmaxf(0.0f, ndoth));
  float res[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float dif = pow_pos(a.diffuse[c * 3 + k], 2.2f);
    const float spc = a.specular ? pow_pos(a.specular[c * 3 + k], 2.2f) : 0.0f;
    const float ambient = a.gi[c * 3 + k] * dif * occ;
    const float dterm = dif * (fmaxf(0.0f, ndotl) * shadow) * a.light_intensity;
    const float sterm = 0.75f * spc * spec_f * shadow;
    const float col = (ambient + dterm + sterm) * a.exposure;
    res[k] = pow_pos(quotient_any(col, 1.0f + col), 1.0f / 2.2f);
  }
  // together, so that no channel's loads wait behind another's store (41.3 ->
  // 37.0 us at 1080p), and as a stream past the L2s (35.6)
  float* o = a.out + c * 3;
  __builtin_nontemporal_store(res[0], o);
  __builtin_nontemporal_store(res[1], o + 1);
  __builtin_nontemporal_store(res[2], o + 2);
}

}  // namespace

hipError_t launch_composite(hipStream_t s, const CompositeArgs& a) {
  const dim3 grid((a.w + 63) / 64, (a.h + 3) / 4);
  hipLaunchKernelGGL(composite_kernel, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

}  // namespace mlgi
