// Ray casting of the procedural scene, shared by the host renderer
// (scene.cpp) and the device renderer (raycast.hip): the same double
// precision code (both compiled with -ffp-contract=off) so that both write
// the same G-buffer and RSM texels.
#pragma once

#include <math.h>
#include <stdint.h>

#if defined(__HIP__)
#include <hip/hip_runtime.h>
#define MLGI_HD __host__ __device__
#else
#define MLGI_HD
#endif

namespace mlgi_scene_impl {

struct D3 {
  double x, y, z;
};
MLGI_HD inline D3 operator+(D3 a, D3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
MLGI_HD inline D3 operator-(D3 a, D3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
MLGI_HD inline D3 operator*(D3 a, double s) { return {a.x * s, a.y * s, a.z * s}; }
MLGI_HD inline double dot(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
MLGI_HD inline D3 cross(D3 a, D3 b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}
MLGI_HD inline double len(D3 a) { return sqrt(dot(a, a)); }
MLGI_HD inline D3 norm(D3 a) { return a * (1.0 / len(a)); }
MLGI_HD inline double comp(D3 a, int i) { return i == 0 ? a.x : (i == 1 ? a.y : a.z); }

struct Tri {
  D3 v0, v1, v2, n;
  float albedo[3];
};

// Binary BVH node of the build (scene.cpp); the ray casters walk the 8-wide
// form below.
struct Node {
  float lo[3], hi[3];
  // leaf: count > 0, left = first index; inner: left child, right = left + 1, count = 0
  int left, count;
};

// 8-wide BVH node: eight child records of 32 bytes, the used ones first. The
// boxes are floats that contain their triangles with a margin (kBoxMargin),
// so that a slab test in FP32 keeps every box the exact ray touches.
struct Child8 {
  float lo[3], hi[3];
  uint32_t ref;  // index << 3 | count: inner child: node index, count 0; leaf child: first triangle
                 // (leaf order), 1..4 triangles; unused: kNoChild, with a box that no ray hits
  // The children's front-to-back order per direction octant, in the eight
  // children's words: octant o (bit a set: the ray runs towards smaller
  // coordinates along axis a) < 4 takes words 2 o (children 0..3) and 2 o + 1
  // (4..7); byte k is the set of children that come after child k. Octant
  // o ^ 7 is the exact reverse.
  uint32_t after;
};
struct alignas(16) Node8 {
  Child8 c[8];
};
constexpr uint32_t kNoChild = 0xFFFFFFFFu;

// Margin of the node boxes, as a share of the scene's largest coordinate
// magnitude m. A ray's FP32 slab distances are off by at most (2^-21 + 2^-22) m
// in position along an axis: the reciprocal direction (rounded direction and
// hardware reciprocal, 2^-22 of a distance of at most 2 m), the rounded origin
// (2^-24 m, the origin moved into the scene's box first: from up to 2^28 m away
// that adds 2^-24 m), its product with the reciprocal (2^-24 m) and the final
// sum (2^-24 of 2 m).
constexpr float kBoxMargin = 0x1p-20f;

// Triangle geometry in leaf order for the intersection test: v0 and the two
// edges v1 - v0, v2 - v0 (computed once, in double, as the test would). The
// array carries three zero entries past the last triangle, so that a leaf's
// four slots can be loaded without a bounds test.
constexpr int kGeoPad = 3;
constexpr int kLeafTris = 4;
struct TriGeo {
  D3 v0, e1, e2;
};

struct Hit {
  double t;
  int tri;
};

// The scene as flat arrays (host vectors or device copies).
struct SceneView {
  const Node8* nodes;  // nodes[0] is the root
  const TriGeo* geo;   // leaf order
  const Tri* tris;     // scene order (normals, albedo, sampling)
  const int* order;    // leaf order -> scene order
  int n_nodes, n_tris;
  float lo[3], hi[3];  // the scene's box, with the nodes' margin
};

// Slab test of a float box in double, without early exits: t0 only grows and
// t1 only shrinks, so testing once after the three axes gives the same answer.
MLGI_HD inline bool box_hit(const float lo_[3], const float hi_[3], D3 o, D3 inv, double tmax, double* tnear) {
  double t0 = 0.0, t1 = tmax;
  for (int k = 0; k < 3; ++k) {
    const double a = ((double)lo_[k] - comp(o, k)) * comp(inv, k);
    const double b = ((double)hi_[k] - comp(o, k)) * comp(inv, k);
    const double lo = (a > b) ? b : a, hi = (a > b) ? a : b;
    t0 = (t0 < lo) ? lo : t0;  // std::max(t0, lo)
    t1 = (hi < t1) ? hi : t1;  // std::min(t1, hi)
  }
  *tnear = t0;
  return !(t0 > t1);
}

MLGI_HD inline D3 ray_inverse(D3 d) {
  return {1.0 / (d.x != 0 ? d.x : 1e-300), 1.0 / (d.y != 0 ? d.y : 1e-300), 1.0 / (d.z != 0 ? d.z : 1e-300)};
}

// A ray for the packets' FP32 box tests: slab distances lo * i + c along each
// axis, measured from the ray's entry into the scene's box (`entry`, 0 for a
// ray that starts inside), and the largest distance still of interest.
struct BoxRay {
  float ix, iy, iz, cx, cy, cz, tmax;
  double entry;
};

// A bound on the distance to t that is not below it (FP32 rounding, 2^-24).
MLGI_HD inline float box_tmax(double t, double entry) { return (float)(t - entry) * (1.0f + 0x1p-22f); }

MLGI_HD inline bool outside_scene(const SceneView& s, D3 o) {
  return !(o.x >= s.lo[0] && o.x <= s.hi[0] && o.y >= s.lo[1] && o.y <= s.hi[1] && o.z >= s.lo[2] && o.z <= s.hi[2]);
}

// 1 / v, finite and not 0 for every v.
MLGI_HD inline float box_inverse(double v) {
  const float f = (float)v;
  const float g = copysignf(fminf(fmaxf(fabsf(f), 1e-18f), 0x1p100f), f);
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_rcpf(g);
#else
  return 1.0f / g;
#endif
}

MLGI_HD inline BoxRay box_ray(D3 o, D3 d, double entry, double tmax, bool in) {
  BoxRay r;
  r.entry = entry;
  const D3 p = o + d * entry;
  r.ix = box_inverse(d.x);
  r.iy = box_inverse(d.y);
  r.iz = box_inverse(d.z);
  r.cx = -((float)p.x * r.ix);
  r.cy = -((float)p.y * r.iy);
  r.cz = -((float)p.z * r.iz);
  // a ray that misses the scene's box, or is not finite (a camera without a far
  // plane, or at its own centre): it enters no box and hits nothing, as on the
  // host. tmax is compared, the distances, which may be NaN, are not.
  const bool finite = fabsf(r.cx) < HUGE_VALF && fabsf(r.cy) < HUGE_VALF && fabsf(r.cz) < HUGE_VALF;
  r.tmax = in && finite ? box_tmax(tmax, entry) : -1.0f;
  return r;
}

// Whether the ray enters the box at most r.tmax away (the distance is
// clamped to 0 and returned). An unused child's box, a point at infinity on
// every axis, is never hit: where tmax is not negative its distances are
// infinite (i is not 0 and c is finite) and tmax is finite.
MLGI_HD inline bool box_test(const BoxRay& r, float lx, float ly, float lz, float hx, float hy, float hz, float& near) {
  const float ax = __builtin_fmaf(lx, r.ix, r.cx), bx = __builtin_fmaf(hx, r.ix, r.cx);
  const float ay = __builtin_fmaf(ly, r.iy, r.cy), by = __builtin_fmaf(hy, r.iy, r.cy);
  const float az = __builtin_fmaf(lz, r.iz, r.cz), bz = __builtin_fmaf(hz, r.iz, r.cz);
  near = fmaxf(fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fminf(az, bz)), 0.0f);
  const float far = fminf(fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz)), r.tmax);
  return near <= far;
}

// Moller-Trumbore, two-sided, in two steps: the determinant and the three
// numerators, then, where tri_maybe has not ruled the triangle out by signs
// and magnitudes alone (no division), the quotients and the exact tests.
struct TriTerms {
  double det, u, v, t;
};
MLGI_HD inline TriTerms tri_terms(const TriGeo& g, D3 o, D3 d) {
  const D3 p = cross(d, g.e2);
  const D3 s = o - g.v0;
  const D3 q = cross(s, g.e1);
  return TriTerms{dot(g.e1, p), dot(s, p), dot(d, q), dot(g.e2, q)};
}
// False only where tri_accept is false: a quotient has the sign of its
// numerator times the determinant's, and one over 1 + 1e-10 (or over
// tmax (1 + 1e-10)) stays over its limit after any rounding.
MLGI_HD inline bool tri_maybe(const TriTerms& k, double tmax) {
  const double a = fabs(k.det);
  const double u = k.det < 0.0 ? -k.u : k.u, v = k.det < 0.0 ? -k.v : k.v, t = k.det < 0.0 ? -k.t : k.t;
  const double lim = a * (1.0 + 1e-10);
  return (a >= 1e-14) & (u >= 0.0) & (v >= 0.0) & (u + v <= lim) & (t > 0.0) & (t <= lim * tmax);
}
// The exact test of a triangle that tri_maybe let through: t in (0, tmax].
MLGI_HD inline bool tri_accept(const TriTerms& k, double tmax, double* th) {
  const double inv = 1.0 / k.det;
  const double u = k.u * inv;
  if (u < 0.0 || u > 1.0) return false;
  const double v = k.v * inv;
  if (v < 0.0 || u + v > 1.0) return false;
  const double tt = k.t * inv;
  if (tt <= 0.0 || tt > tmax) return false;
  *th = tt;
  return true;
}
// Whether a hit of triangle i (leaf order) at t replaces h: the nearer one, of
// equally near ones the first in leaf order, whatever order they were found
// in. A hit at the ray's end is none.
MLGI_HD inline bool hit_before(double t, int i, const Hit& h) { return t < h.t || (t == h.t && i < h.tri); }

// Pending children of a traversal; the build keeps every path's sum of
// (children - 1) below it.
constexpr int kTraceStack = 128;

// A pending child and its box's entry distance.
struct StackEntry {
  uint32_t ref;
  double tnear;
};
struct LocalStack {
  StackEntry e[kTraceStack];
};

// Nearest hit with t < tmax, on the host: an inner node's child boxes are
// tested, the hit ones pushed, farthest first; a popped child is skipped if
// its box is entered beyond the nearest hit so far. The device walks the same
// nodes in packets (raycast.hip). Which of the triangles is nearest, and which
// of equally near ones wins, does not depend on the order of the visits, so
// both give the same hit.
inline Hit trace(const SceneView& s, D3 o, D3 d, double tmax, LocalStack& st) {
  Hit h{tmax, -1};
  const D3 inv = ray_inverse(d);
  int sp = 0;
  uint32_t cur = 0;  // the root, an inner node
  while (true) {
    const int count = (int)(cur & 7u), first = (int)(cur >> 3);
    if (count == 0) {
      const Node8& nd = s.nodes[first];
      const int base = sp;
      for (int k = 0; k < 8 && nd.c[k].ref != kNoChild; ++k) {
        double tn;
        if (!box_hit(nd.c[k].lo, nd.c[k].hi, o, inv, h.t, &tn)) continue;
        int i = sp++;  // insert, the nearest last (never full: see kTraceStack)
        for (; i > base && st.e[i - 1].tnear < tn; --i) st.e[i] = st.e[i - 1];
        st.e[i] = StackEntry{nd.c[k].ref, tn};
      }
    } else {
      for (int k = 0; k < count; ++k) {
        const TriGeo& g = s.geo[first + k];
        const D3 p = cross(d, g.e2), v = o - g.v0;
        const double det = dot(g.e1, p), u = dot(v, p);
        // tri_maybe is false where u alone is out of range: most triangles end
        // here (one thread, 480 x 270 texels: 500 triangles 51.5 -> 49.0 ms,
        // 4,000 111 -> 105, 40,000 156 -> 148)
        if (!((det < 0.0 ? -u : u) >= 0.0) || fabs(u) > fabs(det) * (1.0 + 1e-10)) continue;
        const TriTerms q = tri_terms(g, o, d);
        double th;
        if (tri_maybe(q, h.t) && tri_accept(q, h.t, &th) && hit_before(th, first + k, h)) {
          h.t = th;
          h.tri = first + k;
        }
      }
    }
    do {
      if (sp == 0) {
        if (h.tri >= 0) h.tri = s.order[h.tri];
        return h;
      }
      --sp;
    } while (st.e[sp].tnear > h.t);
    cur = st.e[sp].ref;
  }
}

// One ray per call (the host renderer). The shading functions below call a
// tracer and store only where it says so (the device's packet tracers run
// whole waves, some lanes of which do not store).
struct StackTracer {
  LocalStack st;
  Hit operator()(const SceneView& s, D3 o, D3 d, double tmax) { return trace(s, o, d, tmax, st); }
  bool stores() const { return true; }
};

// 4x4 column-major, double
struct M4 {
  double m[16];
};
MLGI_HD inline void xform(const M4& a, const double v[4], double o[4]) {
  for (int r = 0; r < 4; ++r) {
    double acc = 0;
    for (int c = 0; c < 4; ++c) acc += a.m[c * 4 + r] * v[c];
    o[r] = acc;
  }
}

struct RayCam {
  M4 vp, inv_vp;
  D3 eye, axis;
  double cos_half;  // spot cone (RSM only)
};

// One RSM render of a group (launch_rsms): scene, light, output planes.
struct RsmJob {
  SceneView scene;
  RayCam light;
  float *diffuse, *normal, *depth;
};
constexpr int kRsmJobs = 8;  // per launch: the jobs are kernel arguments (4 KiB)

// Ray through the pixel centre from the near plane to the far plane.
MLGI_HD inline void pixel_ray(const RayCam& rc, int x, int y, int w, int h, D3* o, D3* d) {
  double nx = ((x + 0.5) / w) * 2.0 - 1.0, ny = ((y + 0.5) / h) * 2.0 - 1.0;
  double a[4] = {nx, ny, -1.0, 1.0}, b[4] = {nx, ny, 1.0, 1.0}, pa[4], pb[4];
  xform(rc.inv_vp, a, pa);
  xform(rc.inv_vp, b, pb);
  D3 p0 = {pa[0] / pa[3], pa[1] / pa[3], pa[2] / pa[3]};
  D3 p1 = {pb[0] / pb[3], pb[1] / pb[3], pb[2] / pb[3]};
  *o = p0;
  *d = p1 - p0;
}

MLGI_HD inline double window_depth(const RayCam& rc, D3 p) {
  double v[4] = {p.x, p.y, p.z, 1.0}, c[4];
  xform(rc.vp, v, c);
  return 0.5 * (c[2] / c[3]) + 0.5;
}

// G-buffer texel (x, y): window depth and face normal * 0.5 + 0.5, the
// normal turned towards the viewer; background = depth 1, normal 0.5.
template <class Tracer>
MLGI_HD inline void shade_gbuffer(Tracer& tr, const SceneView& s, const RayCam& rc, int x, int y, int w, int h,
                                  float* depth, float* normal) {
  D3 o, d;
  pixel_ray(rc, x, y, w, h, &o, &d);
  Hit hit = tr(s, o, d, 1.0);
  if (!tr.stores()) return;
  const size_t p = (size_t)y * w + x;
  if (hit.tri < 0) {
    depth[p] = 1.0f;
    normal[p * 3] = normal[p * 3 + 1] = normal[p * 3 + 2] = 0.5f;
    return;
  }
  D3 n = s.tris[hit.tri].n;
  if (dot(n, d) > 0) n = n * -1.0;
  depth[p] = (float)window_depth(rc, o + d * hit.t);
  normal[p * 3 + 0] = (float)n.x * 0.5f + 0.5f;
  normal[p * 3 + 1] = (float)n.y * 0.5f + 0.5f;
  normal[p * 3 + 2] = (float)n.z * 0.5f + 0.5f;
}

// RSM texel (x, y) of a spot light: as the G-buffer, plus the albedo inside
// the cone (0 outside) as the diffuse flux channel.
template <class Tracer>
MLGI_HD inline void shade_rsm(Tracer& tr, const SceneView& s, const RayCam& rc, int x, int y, int w, int h,
                              float* diffuse, float* normal, float* depth) {
  D3 o, d;
  pixel_ray(rc, x, y, w, h, &o, &d);
  Hit hit = tr(s, o, d, 1.0);
  if (!tr.stores()) return;
  const size_t p = (size_t)y * w + x;
  if (hit.tri < 0) {
    depth[p] = 1.0f;
    for (int k = 0; k < 3; ++k) {
      normal[p * 3 + k] = 0.5f;
      diffuse[p * 3 + k] = 0.0f;
    }
    return;
  }
  const Tri& t = s.tris[hit.tri];
  D3 n = t.n;
  if (dot(n, d) > 0) n = n * -1.0;
  const bool in_cone = dot(norm(d), rc.axis) >= rc.cos_half;
  depth[p] = (float)window_depth(rc, o + d * hit.t);
  normal[p * 3 + 0] = (float)n.x * 0.5f + 0.5f;
  normal[p * 3 + 1] = (float)n.y * 0.5f + 0.5f;
  normal[p * 3 + 2] = (float)n.z * 0.5f + 0.5f;
  for (int k = 0; k < 3; ++k) diffuse[p * 3 + k] = in_cone ? t.albedo[k] : 0.0f;
}

// Deferred-shading inputs of texel (x, y) (model.frag:65-132 writes them in
// the reference): the surface albedo (0 for the background) and the VSM
// moments (d, d^2) of the hit's distance d from the camera's eye, which is
// the light's position when rendered from the light (model.frag:130 adds a
// screen-space derivative term to d^2 that a ray caster has no analogue
// of; it is left out). Background: moments (0, 0). Either output may be
// null.
template <class Tracer>
MLGI_HD inline void shade_surface(Tracer& tr, const SceneView& s, const RayCam& rc, int x, int y, int w, int h, float* albedo,
                                  float* moments) {
  D3 o, d;
  pixel_ray(rc, x, y, w, h, &o, &d);
  Hit hit = tr(s, o, d, 1.0);
  if (!tr.stores()) return;
  const size_t p = (size_t)y * w + x;
  if (hit.tri < 0) {
    if (albedo) albedo[p * 3] = albedo[p * 3 + 1] = albedo[p * 3 + 2] = 0.0f;
    if (moments) moments[p * 2] = moments[p * 2 + 1] = 0.0f;
    return;
  }
  if (albedo)
    for (int k = 0; k < 3; ++k) albedo[p * 3 + k] = s.tris[hit.tri].albedo[k];
  if (moments) {
    const double dist = len((o + d * hit.t) - rc.eye);
    moments[p * 2] = (float)dist;
    moments[p * 2 + 1] = (float)(dist * dist);
  }
}

// ------------------------------------------------------------ point sampler
// Area-proportional surface points (the reference's tessellation + geometry
// pass output, ism.tesc:11-23, ism.geom:49-69), shared by the host sampler
// (scene.cpp) and the device sampler (points.hip) so both produce the same
// records. Randomness is counter based: draw k of point i is a splitmix64
// hash of (seed, i, k), so every point is independent of every other.

MLGI_HD inline uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
MLGI_HD inline double counter_uniform(uint64_t seed, uint64_t i, uint64_t k) {
  const uint64_t z = mix64(seed ^ mix64(i * 4 + k + 0x632BE59BD9B4E019ull));
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}
// random.glsl:34-66: random(vec3) = floatConstruct(hash(uvec3 bits))
MLGI_HD inline uint32_t jhash(uint32_t x) {
  x += (x << 10u);
  x ^= (x >> 6u);
  x += (x << 3u);
  x ^= (x >> 11u);
  x += (x << 15u);
  return x;
}
MLGI_HD inline float glsl_random3(float a, float b, float c) {
  uint32_t m = jhash(__builtin_bit_cast(uint32_t, a) ^ jhash(__builtin_bit_cast(uint32_t, b)) ^
                     jhash(__builtin_bit_cast(uint32_t, c)));
  m &= 0x007FFFFFu;
  m |= 0x3F800000u;
  return __builtin_bit_cast(float, m) - 1.0f;
}
// packUnorm4x8 component: round-to-nearest-even of clamp(c, 0, 1) * 255
MLGI_HD inline uint32_t unorm8(float c) {
  const float v = (c < 0.0f ? 0.0f : (c > 1.0f ? 1.0f : c)) * 255.0f;
  return (uint32_t)rintf(v);
}
// std::upper_bound over cdf[0, n): first index with cdf[i] > u
MLGI_HD inline int upper_bound_d(const double* cdf, int n, double u) {
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (cdf[mid] > u)
      hi = mid;
    else
      lo = mid + 1;
  }
  return lo;
}
// Point i: a triangle drawn by area, a uniform point on it, its record
// (pos, packUnorm4x8(n * 0.5 + 0.5, r / 25)) and its bin
// int(random(pos) * n_bins), clamped to [0, n_bins).
// ti: the first triangle whose running area exceeds point_area(), or nt.
MLGI_HD inline double point_area(double total, uint64_t seed, uint64_t i) {
  return counter_uniform(seed, i, 0) * total;
}
MLGI_HD inline void sample_on(const Tri* tris, int ti, int nt, uint64_t seed, uint64_t i, float r_packed, int n_bins,
                              float rec[4], int* bin) {
  if (ti >= nt) ti = nt - 1;
  const Tri& tr = tris[ti];
  const double r1 = sqrt(counter_uniform(seed, i, 1));
  const double r2 = counter_uniform(seed, i, 2);
  const D3 p = tr.v0 * (1.0 - r1) + tr.v1 * (r1 * (1.0 - r2)) + tr.v2 * (r1 * r2);
  const float px = (float)p.x, py = (float)p.y, pz = (float)p.z;
  const uint32_t bits = unorm8((float)tr.n.x * 0.5f + 0.5f) | (unorm8((float)tr.n.y * 0.5f + 0.5f) << 8) |
                        (unorm8((float)tr.n.z * 0.5f + 0.5f) << 16) | (unorm8(r_packed) << 24);
  rec[0] = px;
  rec[1] = py;
  rec[2] = pz;
  rec[3] = __builtin_bit_cast(float, bits);
  const int bi = (int)(glsl_random3(px, py, pz) * (float)n_bins);
  *bin = bi < 0 ? 0 : (bi > n_bins - 1 ? n_bins - 1 : bi);
}
MLGI_HD inline void sample_point(const Tri* tris, const double* cdf, int nt, double total, uint64_t seed,
                                 uint64_t i, float r_packed, int n_bins, float rec[4], int* bin) {
  sample_on(tris, upper_bound_d(cdf, nt, point_area(total, seed, i)), nt, seed, i, r_packed, n_bins, rec, bin);
}

}  // namespace mlgi_scene_impl

struct mlgi_scene;
// Host-side access for the device uploader (scene.cpp).
mlgi_scene_impl::SceneView mlgi_scene_view(const mlgi_scene* s);
// Ray camera of a camera / light: view-projection and inverse (double),
// eye, view axis, cos of the half cone angle.
bool mlgi_scene_ray_cam(const struct mlgi_camera* cam, mlgi_scene_impl::RayCam* out);
// inverse(bias * P * V) of a light as floats (column-major).
bool mlgi_scene_inv_biased_vp(const struct mlgi_camera* light, float* out16);
// Running triangle areas (cdf[i] = sum of areas 0..i, in order); returns the total.
double mlgi_scene_area_cdf(const mlgi_scene* s, double* cdf);
// Packed point radius r / 25 for n points standing for ism_count points each.
float mlgi_scene_point_radius(double total_area, int64_t n_points, int32_t ism_count);
