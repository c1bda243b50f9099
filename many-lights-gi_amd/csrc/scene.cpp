// Host-side synthetic inputs (include/mlgi_scene.h): a seeded procedural
// scene, a BVH ray caster that writes the G-buffer and RSM in the formats the
// reference rasteriser produces (RasterizationStage.cpp:139-149,
// model.frag:93 faceNormal = N*0.5+0.5), and the area-proportional splat
// point set with the reference's point record and bin hash (ism.geom:49-68,
// random.glsl:34-66). Deterministic for a given seed and independent of the
// thread count.
#include <algorithm>
#include <cstdlib>
#include <cmath>
#include <cstring>
#include <thread>
#include <vector>

#include "../../include/mlgi.h"
#include "../../include/mlgi_scene.h"
#include "scene_trace.hpp"

namespace {

using namespace mlgi_scene_impl;

// splitmix64 sequential generator (mix64 and the counter-based draws of the
// point sampler are in scene_trace.hpp)
struct Rng {
  uint64_t s;
  explicit Rng(uint64_t seed) : s(seed) {}
  double uniform() {
    s += 0x9E3779B97F4A7C15ull;
    return (double)(mix64(s) >> 11) * (1.0 / 9007199254740992.0);
  }
};
}  // namespace

struct mlgi_scene {
  std::vector<Tri> tris;
  std::vector<int> order;  // BVH leaf order
  std::vector<Node8> nodes;  // 8-wide BVH
  std::vector<TriGeo> geo;   // triangle geometry in leaf order
  float lo[3], hi[3];        // the scene's box, with the nodes' margin
  double area = 0.0;
};

namespace {

const D3 kDefaultEye = {5.0, 5.0, 9.0};

// Float bounds that contain the double ones.
float round_up_f(double x) {
  float f = (float)x;
  if ((double)f < x) f = std::nextafter(f, HUGE_VALF);
  return f;
}
float round_down_f(double x) {
  float f = (float)x;
  if ((double)f > x) f = std::nextafter(f, -HUGE_VALF);
  return f;
}

struct Box {
  float lo[3], hi[3];
  void clear() {
    for (int k = 0; k < 3; ++k) lo[k] = HUGE_VALF, hi[k] = -HUGE_VALF;
  }
  void add(const float* l, const float* h) {
    for (int k = 0; k < 3; ++k) {
      lo[k] = l[k] < lo[k] ? l[k] : lo[k];
      hi[k] = h[k] > hi[k] ? h[k] : hi[k];
    }
  }
  float area() const {
    const float x = hi[0] - lo[0], y = hi[1] - lo[1], z = hi[2] - lo[2];
    return x < 0.0f ? 0.0f : x * y + y * z + z * x;
  }
};

// A triangle as the build sees it: its box (floats, rounded outward) and twice
// its centre.
struct Prim {
  float lo[3], hi[3], c[3];
  int tri;
};

// The binary tree over prims (reordered into leaf order): binned surface-area
// splits down to depth sah_depth, median splits below it and wherever no
// binned split separates; leaves of at most kLeafTris triangles.
void build_binary(std::vector<Prim>& prims, float span, int sah_depth, std::vector<Node>& nodes) {
  const int n = (int)prims.size();
  nodes.clear();
  nodes.reserve(n + 8);
  nodes.push_back(Node{});
  struct Item {
    int node, begin, end, depth;
  };
  std::vector<Item> stack;
  // Root split by size: triangles spanning more than a quarter of the scene
  // (the room's walls) go to their own subtree, so the boxes of the splits
  // below stay tight around the small geometry instead of every level
  // containing a wall (which each ray would then enter).
  auto big = [&](const Prim& p) {
    for (int k = 0; k < 3; ++k)
      if (p.hi[k] - p.lo[k] > 0.25f * span) return true;
    return false;
  };
  const int n_big = (int)(std::stable_partition(prims.begin(), prims.end(), big) - prims.begin());
  auto inner = [&](int node, int begin, int mid, int end, int depth) {
    nodes[node].left = (int)nodes.size();
    nodes[node].count = 0;
    const int left = nodes[node].left;
    nodes.push_back(Node{});
    nodes.push_back(Node{});
    stack.push_back({left, begin, mid, depth + 1});
    stack.push_back({left + 1, mid, end, depth + 1});
  };
  if (n_big > 0 && n_big < n && n > kLeafTris) {
    Box b;
    b.clear();
    for (const Prim& p : prims) b.add(p.lo, p.hi);
    std::copy(b.lo, b.lo + 3, nodes[0].lo);
    std::copy(b.hi, b.hi + 3, nodes[0].hi);
    inner(0, 0, n_big, n, 0);
  } else {
    stack.push_back({0, 0, n, 0});
  }
  while (!stack.empty()) {
    const Item it = stack.back();
    stack.pop_back();
    const int cnt = it.end - it.begin;
    Prim* const p0 = prims.data() + it.begin;
    Box b;
    b.clear();
    float clo[3] = {HUGE_VALF, HUGE_VALF, HUGE_VALF}, chi[3] = {-HUGE_VALF, -HUGE_VALF, -HUGE_VALF};
    for (int i = 0; i < cnt; ++i) {
      b.add(p0[i].lo, p0[i].hi);
      for (int k = 0; k < 3; ++k) {
        clo[k] = std::min(clo[k], p0[i].c[k]);
        chi[k] = std::max(chi[k], p0[i].c[k]);
      }
    }
    std::copy(b.lo, b.lo + 3, nodes[it.node].lo);
    std::copy(b.hi, b.hi + 3, nodes[it.node].hi);
    if (cnt <= kLeafTris) {
      nodes[it.node].left = it.begin;
      nodes[it.node].count = cnt;
      continue;
    }
    // Binned surface-area heuristic: centroid bins per axis (as many as
    // triangles in small nodes), the plane of least (area x count) over both
    // sides.
    constexpr int kBins = 16;
    const int nb = std::min(kBins, std::max(4, cnt));
    int axis = -1, split = -1;
    float scale[3];
    auto bin_of = [&](const Prim& p, int k) { return std::min(nb - 1, (int)((p.c[k] - clo[k]) * scale[k])); };
    if (it.depth < sah_depth) {
      Box bx[3][kBins];
      int bc[3][kBins];
      for (int k = 0; k < 3; ++k) {
        scale[k] = chi[k] > clo[k] ? (float)nb / (chi[k] - clo[k]) : 0.0f;
        if (!(scale[k] < HUGE_VALF)) scale[k] = 0.0f;
        for (int q = 0; q < nb; ++q) {
          bx[k][q].clear();
          bc[k][q] = 0;
        }
      }
      for (int i = 0; i < cnt; ++i)
        for (int k = 0; k < 3; ++k) {
          const int q = bin_of(p0[i], k);
          bx[k][q].add(p0[i].lo, p0[i].hi);
          bc[k][q]++;
        }
      float best = HUGE_VALF;
      for (int k = 0; k < 3; ++k) {
        float right[kBins];  // area x count of bins [q, nb)
        Box acc;
        acc.clear();
        int rc = 0;
        for (int q = nb - 1; q >= 1; --q) {
          acc.add(bx[k][q].lo, bx[k][q].hi);
          rc += bc[k][q];
          right[q] = acc.area() * (float)rc;
        }
        acc.clear();
        int lc = 0;
        for (int q = 1; q < nb; ++q) {  // left = bins [0, q)
          acc.add(bx[k][q - 1].lo, bx[k][q - 1].hi);
          lc += bc[k][q - 1];
          if (lc == 0 || lc == cnt) continue;
          const float cost = acc.area() * (float)lc + right[q];
          if (cost < best) {
            best = cost;
            axis = k;
            split = q;
          }
        }
      }
    }
    int mid = 0;
    if (axis >= 0) {
      const int ax = axis, spl = split;
      mid = (int)(std::partition(p0, p0 + cnt, [&](const Prim& p) { return bin_of(p, ax) < spl; }) - p0);
    }
    if (mid <= 0 || mid >= cnt) {
      axis = 0;
      for (int k = 1; k < 3; ++k)
        if (chi[k] - clo[k] > chi[axis] - clo[axis]) axis = k;
      mid = cnt / 2;
      std::nth_element(p0, p0 + mid, p0 + cnt, [axis](const Prim& a, const Prim& c) {
        return a.c[axis] < c.c[axis] || (a.c[axis] == c.c[axis] && a.tri < c.tri);
      });
    }
    inner(it.node, it.begin, it.begin + mid, it.end, it.depth);
  }
}

// 8-wide node of binary node b: the child of largest area is opened until
// eight are there (levels: the children of three binary levels, opened
// whatever their area, which bounds the depth). Returns the most children
// that can be pending below it (kTraceStack).
int collapse8(mlgi_scene* s, const std::vector<Node>& bin, int b, float margin, bool levels) {
  const int me = (int)s->nodes.size();
  s->nodes.push_back(Node8{});
  int kid[8] = {b}, depth[8] = {0}, n = 1;
  auto area = [&](int x) {
    Box q;
    std::copy(bin[x].lo, bin[x].lo + 3, q.lo);
    std::copy(bin[x].hi, bin[x].hi + 3, q.hi);
    return q.area();
  };
  while (n < 8) {
    int open = -1;
    float best = -1.0f;
    for (int k = 0; k < n; ++k) {
      if (bin[kid[k]].count > 0 || (levels && depth[k] == 3)) continue;
      const float a = levels ? 8.0f - (float)depth[k] : area(kid[k]);
      if (a > best) best = a, open = k;
    }
    if (open < 0) break;
    const int left = bin[kid[open]].left;
    depth[n] = ++depth[open];
    kid[open] = left;
    kid[n++] = left + 1;
  }
  Node8 q;
  float centre[8][3];
  int most = 0;
  for (int k = 0; k < 8; ++k) {
    Child8& c = q.c[k];
    c.after = 0;
    if (k >= n) {
      c.ref = kNoChild;
      // a point no ray reaches (box_test): the slab test sorts each axis's two
      // planes, so an inverted box would count as an endless one
      for (int a = 0; a < 3; ++a) c.lo[a] = c.hi[a] = HUGE_VALF;
      continue;
    }
    const Node& x = bin[kid[k]];
    for (int a = 0; a < 3; ++a) {
      c.lo[a] = round_down_f((double)x.lo[a] - margin);
      c.hi[a] = round_up_f((double)x.hi[a] + margin);
      centre[k][a] = 0.5f * x.lo[a] + 0.5f * x.hi[a];
    }
    if (x.count > 0) {
      c.ref = (uint32_t)x.left << 3 | (uint32_t)x.count;
    } else {
      c.ref = (uint32_t)s->nodes.size() << 3;
      most = std::max(most, collapse8(s, bin, kid[k], margin, levels));
    }
  }
  // children by their centres' distance along the octant's diagonal
  for (int o = 0; o < 4; ++o) {
    float key[8];
    for (int k = 0; k < n; ++k) {
      key[k] = 0.0f;
      for (int a = 0; a < 3; ++a) key[k] += (o >> a & 1) ? -centre[k][a] : centre[k][a];
    }
    uint32_t word[2] = {0, 0};
    for (int k = 0; k < n; ++k)
      for (int j = 0; j < n; ++j)
        if (key[j] > key[k] || (key[j] == key[k] && j > k)) word[k >> 2] |= (1u << j) << (8 * (k & 3));
    q.c[2 * o].after = word[0];
    q.c[2 * o + 1].after = word[1];
  }
  s->nodes[me] = q;
  return most + n - 1;
}

// Binned splits throughout; if the tree could outgrow the traversal stack
// (only for far larger scenes than generated here), median splits and whole
// levels: at most 7 pending children for each three binary levels, of which
// median splits make ceil(log2(n / 4)) + 2 <= 31. Then the triangle geometry
// in leaf order. False where neither tree stays below `stack` pending children
// (not for kTraceStack).
bool build_bvh(mlgi_scene* s, int stack = kTraceStack) {
  const int n = (int)s->tris.size();
  std::vector<Prim> prims(n);
  Box scene;
  scene.clear();
  for (int i = 0; i < n; ++i) {
    const Tri& t = s->tris[i];
    Prim& p = prims[i];
    p.tri = i;
    for (int k = 0; k < 3; ++k) {
      const double a = comp(t.v0, k), b = comp(t.v1, k), c = comp(t.v2, k);
      p.lo[k] = round_down_f(std::min(a, std::min(b, c)));
      p.hi[k] = round_up_f(std::max(a, std::max(b, c)));
      p.c[k] = p.lo[k] + p.hi[k];
    }
    scene.add(p.lo, p.hi);
  }
  float span = 0.0f, mag = 0.0f;
  for (int k = 0; k < 3; ++k) {
    span = std::max(span, scene.hi[k] - scene.lo[k]);
    mag = std::max(mag, std::max(std::fabs(scene.lo[k]), std::fabs(scene.hi[k])));
  }
  const float margin = mag * kBoxMargin;
  for (int k = 0; k < 3; ++k) {
    s->lo[k] = round_down_f((double)scene.lo[k] - margin);
    s->hi[k] = round_up_f((double)scene.hi[k] + margin);
  }
  std::vector<Node> bin;
  bool fits = false;
  for (int levels = 0; levels < 2 && !fits; ++levels) {
    build_binary(prims, span, levels ? 0 : 64, bin);
    s->nodes.clear();
    fits = collapse8(s, bin, 0, margin, levels != 0) < stack;
  }
  if (!fits) return false;
  s->order.resize(n);
  s->geo.assign(n + kGeoPad, TriGeo{});
  for (int i = 0; i < n; ++i) {
    s->order[i] = prims[i].tri;
    const Tri& t = s->tris[s->order[i]];
    s->geo[i] = TriGeo{t.v0, t.v1 - t.v0, t.v2 - t.v0};
  }
  return true;
}

// 4x4 column-major helpers in double
M4 mul(const M4& a, const M4& b) {
  M4 r{};
  for (int c = 0; c < 4; ++c)
    for (int rr = 0; rr < 4; ++rr) {
      double acc = 0;
      for (int k = 0; k < 4; ++k) acc += a.m[k * 4 + rr] * b.m[c * 4 + k];
      r.m[c * 4 + rr] = acc;
    }
  return r;
}
bool inverse(const M4& a, M4* out) {
  double m[4][8];
  for (int r = 0; r < 4; ++r)
    for (int c = 0; c < 4; ++c) {
      m[r][c] = a.m[c * 4 + r];
      m[r][c + 4] = r == c ? 1.0 : 0.0;
    }
  for (int c = 0; c < 4; ++c) {
    int piv = c;
    for (int r = c + 1; r < 4; ++r)
      if (std::fabs(m[r][c]) > std::fabs(m[piv][c])) piv = r;
    if (std::fabs(m[piv][c]) < 1e-300) return false;
    for (int k = 0; k < 8; ++k) std::swap(m[c][k], m[piv][k]);
    double d = m[c][c];
    for (int k = 0; k < 8; ++k) m[c][k] /= d;
    for (int r = 0; r < 4; ++r) {
      if (r == c) continue;
      double f = m[r][c];
      for (int k = 0; k < 8; ++k) m[r][k] -= f * m[c][k];
    }
  }
  for (int r = 0; r < 4; ++r)
    for (int c = 0; c < 4; ++c) out->m[c * 4 + r] = m[r][c + 4];
  return true;
}
void camera_matrices(const mlgi_camera* cam, M4* view, M4* proj) {
  D3 eye = {cam->eye[0], cam->eye[1], cam->eye[2]};
  D3 ctr = {cam->center[0], cam->center[1], cam->center[2]};
  D3 up = {cam->up[0], cam->up[1], cam->up[2]};
  D3 f = norm(ctr - eye);
  D3 s = norm(cross(f, up));
  D3 u = cross(s, f);
  M4 v{};
  v.m[0] = s.x; v.m[4] = s.y; v.m[8] = s.z;
  v.m[1] = u.x; v.m[5] = u.y; v.m[9] = u.z;
  v.m[2] = -f.x; v.m[6] = -f.y; v.m[10] = -f.z;
  v.m[12] = -dot(s, eye); v.m[13] = -dot(u, eye); v.m[14] = dot(f, eye);
  v.m[15] = 1.0;
  *view = v;
  const double th = std::tan((double)cam->fovy_deg * M_PI / 180.0 / 2.0);
  const double n = cam->z_near, fa = cam->z_far;
  M4 p{};
  p.m[0] = 1.0 / ((double)cam->aspect * th);
  p.m[5] = 1.0 / th;
  p.m[10] = -(fa + n) / (fa - n);
  p.m[11] = -1.0;
  p.m[14] = -(2.0 * fa * n) / (fa - n);
  *proj = p;
}

void to_float(const M4& a, float* o) {
  for (int i = 0; i < 16; ++i) o[i] = (float)a.m[i];
}

// Worker threads of the host renderer and sampler: `t` when positive, else
// OMP_NUM_THREADS when set (the process's share of the host), else the
// hardware's thread count (at most 64).
int nthreads(int t) {
  if (t > 0) return t;
  if (const char* e = std::getenv("OMP_NUM_THREADS")) {
    const int n = std::atoi(e);
    if (n > 0) return std::min(n, 64);
  }
  unsigned h = std::thread::hardware_concurrency();
  return h ? (int)std::min(h, 64u) : 4;
}

template <class F>
void parallel_rows(int rows, int threads, F f) {
  const int nt = std::max(1, std::min(threads, rows));
  std::vector<std::thread> pool;
  for (int t = 0; t < nt; ++t)
    pool.emplace_back([=]() {
      for (int y = t; y < rows; y += nt) f(y);
    });
  for (auto& th : pool) th.join();
}

RayCam ray_cam(const mlgi_camera* cam) {
  M4 v, p;
  camera_matrices(cam, &v, &p);
  RayCam rc;
  rc.vp = mul(p, v);
  inverse(rc.vp, &rc.inv_vp);
  rc.eye = {cam->eye[0], cam->eye[1], cam->eye[2]};
  rc.axis = norm(D3{cam->center[0], cam->center[1], cam->center[2]} - rc.eye);
  rc.cos_half = std::cos((double)cam->fovy_deg * M_PI / 180.0 / 2.0);
  return rc;
}

SceneView view_of(const mlgi_scene* s);

}  // namespace

extern "C" {

int mlgi_scene_create(uint64_t seed, int32_t n_random, mlgi_scene** out) {
  if (!out || n_random < 0) return MLGI_ERR_INVALID_ARGUMENT;
  auto* s = new mlgi_scene();
  Rng rng(seed);
  const double L = 10.0;
  auto quad = [&](D3 a, D3 b, D3 c, D3 d, D3 n) {
    for (int k = 0; k < 2; ++k) {
      Tri t;
      t.v0 = a;
      t.v1 = k == 0 ? b : c;
      t.v2 = k == 0 ? c : d;
      t.n = n;
      for (int i = 0; i < 3; ++i) t.albedo[i] = (float)(0.2 + 0.6 * rng.uniform());
      s->tris.push_back(t);
    }
  };
  quad({0, 0, 0}, {L, 0, 0}, {L, 0, L}, {0, 0, L}, {0, 1, 0});    // floor
  quad({0, L, 0}, {L, L, 0}, {L, L, L}, {0, L, L}, {0, -1, 0});   // ceiling
  quad({0, 0, 0}, {0, L, 0}, {0, L, L}, {0, 0, L}, {1, 0, 0});    // x = 0
  quad({L, 0, 0}, {L, L, 0}, {L, L, L}, {L, 0, L}, {-1, 0, 0});   // x = L
  quad({0, 0, 0}, {L, 0, 0}, {L, L, 0}, {0, L, 0}, {0, 0, 1});    // z = 0
  quad({0, 0, L}, {L, 0, L}, {L, L, L}, {0, L, L}, {0, 0, -1});   // z = L
  auto dir = [&]() {
    double z = 2.0 * rng.uniform() - 1.0, ph = 2.0 * M_PI * rng.uniform();
    double r = std::sqrt(std::max(0.0, 1.0 - z * z));
    return D3{r * std::cos(ph), r * std::sin(ph), z};
  };
  int made = 0;
  while (made < n_random) {
    D3 v0 = {0.5 + 9.0 * rng.uniform(), 0.5 + 9.0 * rng.uniform(), 0.5 + 9.0 * rng.uniform()};
    D3 e1 = dir() * (0.1 + 0.4 * rng.uniform());
    D3 e2 = dir() * (0.1 + 0.4 * rng.uniform());
    float alb[3];
    for (int i = 0; i < 3; ++i) alb[i] = (float)(0.2 + 0.6 * rng.uniform());
    D3 c = cross(e1, e2);
    if (len(c) < 1e-4) continue;
    if (len(v0 - kDefaultEye) < 1.0) continue;  // keep the default camera clear
    Tri t;
    t.v0 = v0;
    t.v1 = v0 + e1;
    t.v2 = v0 + e2;
    t.n = norm(c);
    std::memcpy(t.albedo, alb, sizeof alb);
    s->tris.push_back(t);
    ++made;
  }
  for (const Tri& t : s->tris) s->area += 0.5 * len(cross(t.v1 - t.v0, t.v2 - t.v0));
  if (!build_bvh(s)) {
    delete s;
    return MLGI_ERR_UNSUPPORTED;
  }
  *out = s;
  return MLGI_OK;
}

void mlgi_scene_destroy(mlgi_scene* s) { delete s; }

int32_t mlgi_scene_triangle_count(const mlgi_scene* s) { return s ? (int32_t)s->tris.size() : 0; }

double mlgi_scene_total_area(const mlgi_scene* s) { return s ? s->area : 0.0; }

int mlgi_scene_triangles(const mlgi_scene* s, float* v, float* n, float* a) {
  if (!s) return MLGI_ERR_INVALID_ARGUMENT;
  for (size_t i = 0; i < s->tris.size(); ++i) {
    const Tri& t = s->tris[i];
    if (v) {
      const D3* p[3] = {&t.v0, &t.v1, &t.v2};
      for (int k = 0; k < 3; ++k) {
        v[i * 9 + k * 3 + 0] = (float)p[k]->x;
        v[i * 9 + k * 3 + 1] = (float)p[k]->y;
        v[i * 9 + k * 3 + 2] = (float)p[k]->z;
      }
    }
    if (n) {
      n[i * 3 + 0] = (float)t.n.x;
      n[i * 3 + 1] = (float)t.n.y;
      n[i * 3 + 2] = (float)t.n.z;
    }
    if (a) std::memcpy(a + i * 3, t.albedo, sizeof t.albedo);
  }
  return MLGI_OK;
}

void mlgi_scene_default_camera(float aspect, mlgi_camera* c) {
  if (!c) return;
  const float eye[3] = {(float)kDefaultEye.x, (float)kDefaultEye.y, (float)kDefaultEye.z};
  const float ctr[3] = {5.0f, 4.0f, 0.0f};
  const float up[3] = {0.0f, 1.0f, 0.0f};
  std::memcpy(c->eye, eye, sizeof eye);
  std::memcpy(c->center, ctr, sizeof ctr);
  std::memcpy(c->up, up, sizeof up);
  c->fovy_deg = 60.0f;
  c->aspect = aspect;
  c->z_near = 0.05f;
  c->z_far = 50.0f;
}

void mlgi_scene_light_pose(uint64_t seed, mlgi_camera* c) {
  if (!c) return;
  Rng rng(seed ^ 0x5107A11C0FFEEull);
  c->eye[0] = (float)(2.0 + 6.0 * rng.uniform());
  c->eye[1] = (float)(8.5 + 1.0 * rng.uniform());
  c->eye[2] = (float)(2.0 + 6.0 * rng.uniform());
  c->center[0] = (float)(1.0 + 8.0 * rng.uniform());
  c->center[1] = (float)(0.0 + 2.0 * rng.uniform());
  c->center[2] = (float)(1.0 + 8.0 * rng.uniform());
  c->up[0] = 0.0f;
  c->up[1] = 0.0f;
  c->up[2] = 1.0f;
  c->fovy_deg = 45.0f;
  c->aspect = 1.0f;
  c->z_near = 0.05f;
  c->z_far = 50.0f;
}

int mlgi_camera_matrices(const mlgi_camera* cam, float* view16, float* proj16, float* vp_inv16) {
  if (!cam) return MLGI_ERR_INVALID_ARGUMENT;
  M4 v, p;
  camera_matrices(cam, &v, &p);
  if (view16) to_float(v, view16);
  if (proj16) to_float(p, proj16);
  if (vp_inv16) {
    M4 inv;
    if (!inverse(mul(p, v), &inv)) return MLGI_ERR_INVALID_ARGUMENT;
    to_float(inv, vp_inv16);
  }
  return MLGI_OK;
}

int mlgi_scene_render_gbuffer(const mlgi_scene* s, const mlgi_camera* cam, int32_t w, int32_t h,
                              int32_t threads, float* depth, float* normal) {
  if (!s || !cam || w <= 0 || h <= 0 || !depth || !normal) return MLGI_ERR_INVALID_ARGUMENT;
  const RayCam rc = ray_cam(cam);
  const SceneView sv = view_of(s);
  parallel_rows(h, nthreads(threads), [&](int y) {
    StackTracer tr;
    for (int x = 0; x < w; ++x) shade_gbuffer(tr, sv, rc, x, y, w, h, depth, normal);
  });
  return MLGI_OK;
}

int mlgi_scene_render_rsm(const mlgi_scene* s, const mlgi_camera* light, int32_t w, int32_t h,
                          int32_t threads, float* diffuse, float* normal, float* depth,
                          float* inv_bvp16) {
  if (!s || !light || w <= 0 || h <= 0 || !diffuse || !normal || !depth)
    return MLGI_ERR_INVALID_ARGUMENT;
  const RayCam rc = ray_cam(light);
  const SceneView sv = view_of(s);
  parallel_rows(h, nthreads(threads), [&](int y) {
    StackTracer tr;
    for (int x = 0; x < w; ++x) shade_rsm(tr, sv, rc, x, y, w, h, diffuse, normal, depth);
  });
  if (inv_bvp16 && !mlgi_scene_inv_biased_vp(light, inv_bvp16)) return MLGI_ERR_INVALID_ARGUMENT;
  return MLGI_OK;
}

int mlgi_scene_render_surface(const mlgi_scene* s, const mlgi_camera* cam, int32_t w, int32_t h, int32_t threads,
                              float* albedo, float* moments) {
  if (!s || !cam || w <= 0 || h <= 0 || (!albedo && !moments)) return MLGI_ERR_INVALID_ARGUMENT;
  const RayCam rc = ray_cam(cam);
  const SceneView sv = view_of(s);
  parallel_rows(h, nthreads(threads), [&](int y) {
    StackTracer tr;
    for (int x = 0; x < w; ++x) shade_surface(tr, sv, rc, x, y, w, h, albedo, moments);
  });
  return MLGI_OK;
}

}  // extern "C"

double mlgi_scene_area_cdf(const mlgi_scene* s, double* cdf) {
  double acc = 0.0;
  for (size_t i = 0; i < s->tris.size(); ++i) {
    const Tri& t = s->tris[i];
    acc += 0.5 * len(cross(t.v1 - t.v0, t.v2 - t.v0));
    cdf[i] = acc;
  }
  return acc;
}

float mlgi_scene_point_radius(double total_area, int64_t n_points, int32_t ism_count) {
  // each point stands for ism_count points: radius boosted by sqrt(ism_count) (ism.geom:60-63)
  const double r_world = std::sqrt(total_area / ((double)std::max<int64_t>(n_points, 1) * M_PI)) *
                         std::sqrt((double)ism_count);
  return (float)(r_world / 25.0);
}

extern "C" int mlgi_scene_sample_points(const mlgi_scene* s, int64_t n_points, int32_t n_bins,
                                        int32_t ism_count, uint64_t seed, int32_t threads,
                                        float* records, uint32_t* bin_offsets) {
  if (!s || n_points < 0 || n_points > (1ll << 31) - 1 || n_bins <= 0 || ism_count <= 0 ||
      (!records && n_points) || !bin_offsets)
    return MLGI_ERR_INVALID_ARGUMENT;
  const size_t nt = s->tris.size();
  std::vector<double> cdf(nt);
  const double total = mlgi_scene_area_cdf(s, cdf.data());
  const float r_packed = mlgi_scene_point_radius(total, n_points, ism_count);
  std::vector<float> tmp((size_t)n_points * 4);
  std::vector<int32_t> bin((size_t)n_points);
  const int nth = nthreads(threads);
  const int64_t chunk = (n_points + nth - 1) / std::max(nth, 1);
  std::vector<std::thread> pool;
  for (int t = 0; t < nth; ++t) {
    pool.emplace_back([&, t]() {
      const int64_t b = t * chunk, e = std::min<int64_t>(n_points, b + chunk);
      for (int64_t i = b; i < e; ++i)
        sample_point(s->tris.data(), cdf.data(), (int)nt, total, seed, (uint64_t)i, r_packed, n_bins, &tmp[i * 4],
                     &bin[i]);
    });
  }
  for (auto& th : pool) th.join();
  std::vector<uint32_t> cnt(n_bins + 1, 0);
  for (int64_t i = 0; i < n_points; ++i) cnt[bin[i] + 1]++;
  for (int b = 0; b < n_bins; ++b) cnt[b + 1] += cnt[b];
  std::memcpy(bin_offsets, cnt.data(), sizeof(uint32_t) * (n_bins + 1));
  std::vector<uint32_t> pos(cnt.begin(), cnt.end() - 1);
  for (int64_t i = 0; i < n_points; ++i) {
    uint32_t dst = pos[bin[i]]++;
    std::memcpy(records + (size_t)dst * 4, &tmp[i * 4], 16);
  }
  return MLGI_OK;
}

namespace {
SceneView view_of(const mlgi_scene* s) {
  return SceneView{s->nodes.data(), s->geo.data(), s->tris.data(), s->order.data(), (int)s->nodes.size(),
                   (int)s->tris.size(), {s->lo[0], s->lo[1], s->lo[2]}, {s->hi[0], s->hi[1], s->hi[2]}};
}
}  // namespace

SceneView mlgi_scene_view(const mlgi_scene* s) { return view_of(s); }

bool mlgi_scene_ray_cam(const mlgi_camera* cam, RayCam* out) {
  if (!cam || !out) return false;
  *out = ray_cam(cam);
  return true;
}

bool mlgi_scene_inv_biased_vp(const mlgi_camera* light, float* out16) {
  const RayCam rc = ray_cam(light);
  M4 bias{};
  bias.m[0] = 0.5; bias.m[5] = 0.5; bias.m[10] = 0.5;
  bias.m[12] = 0.5; bias.m[13] = 0.5; bias.m[14] = 0.5; bias.m[15] = 1.0;
  M4 inv;
  if (!inverse(mul(bias, rc.vp), &inv)) return false;
  to_float(inv, out16);
  return true;
}
