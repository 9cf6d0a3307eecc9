// Host check of the forms the four-wide walk reads (pyradiance_amd/csrc):
// 64-byte nodes against the nodes they are rounded from, and leaf records
// against the primitive tables.
#include <algorithm>
#include <cmath>
#include <random>
#include <utility>
#include <vector>

#include "rg_bvh.hpp"

// Random nodes of `nused` children with extents from 1e-5 to 1e4 around
// origins up to `far`: every rounded box holds the box it stands for in exact
// arithmetic, is at most two steps wider on each side, and unused slots hold
// no box.  Returns 0 or a bit mask.
extern "C" int check_quantized(int n, unsigned seed, int nused, double far) {
  std::mt19937 rng(seed);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  std::vector<rg::BVH4Node> in((size_t)n);
  for (auto& N : in) {
    float* lo[3] = {N.lox, N.loy, N.loz};
    float* hi[3] = {N.hix, N.hiy, N.hiz};
    for (int a = 0; a < 3; ++a) {
      const double o = (2 * U(rng) - 1) * far, e = std::pow(10.0, -5 + 9 * U(rng));
      for (int k = 0; k < 4; ++k) {
        const double x = o + e * U(rng);
        lo[a][k] = k < nused ? (float)x : 0.f;
        hi[a][k] = k < nused ? std::nextafter((float)(x + e * U(rng) * U(rng)), INFINITY) : 0.f;
      }
    }
    for (int k = 0; k < 4; ++k) N.child[k] = k < nused ? (int)(rng() & 0xffff) - 0x7fff : INT32_MIN;
    for (int& p : N.pad) p = 0;
  }
  int bad = 0;
  for (size_t i = 0; i < in.size(); ++i) {
    const rg::BVH4Node& N = in[i];
    const rg::BVH4Q Q = rg::quantize_node(N);
    const float* lo[3] = {N.lox, N.loy, N.loz};
    const float* hi[3] = {N.hix, N.hiy, N.hiz};
    const uint32_t ql[3] = {Q.lox, Q.loy, Q.loz}, qh[3] = {Q.hix, Q.hiy, Q.hiz};
    for (int k = 0; k < 4; ++k) {
      if (Q.child[k] != N.child[k]) bad |= 2;
      for (int a = 0; a < 3; ++a) {
        const int l = (ql[a] >> (8 * k)) & 255, h = (qh[a] >> (8 * k)) & 255;
        if (k >= nused) { if (l != 255 || h != 0) bad |= 4; continue; }
        const double s = Q.scale[a], o = Q.org[a];
        if (o + l * s > (double)lo[a][k] || o + h * s < (double)hi[a][k]) bad |= 8;
        if (o + (l + 2) * s < (double)lo[a][k] || o + (h - 2) * s > (double)hi[a][k]) bad |= 16;
      }
    }
  }
  return bad;
}

// Random polygons of nv vertices in planes across each axis (convex and not,
// and with repeated vertices), rays through points inside, outside, on and
// within 3e-6 of edges and vertices: hit_leaf() accepts what hit_prim()
// accepts, with the same distance, orientation and index, from an empty hit
// and from one at a nearly equal distance.  Returns the number of rays that
// differ, and in *hits the number that hit.
extern "C" long check_leaf(int n, int nrays, unsigned seed, int nv, int degenerate, long* hits) {
  using namespace rg;
  std::mt19937 rng(seed);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  long bad = 0, nhit = 0;
  for (int i = 0; i < n; ++i) {
    // vertices on a plane x[ax] = c + s . (the other two), at random in a box
    const int ax = (int)(rng() % 3);
    const double size = std::pow(10.0, -2 + 3 * U(rng)), c = U(rng) * 10 - 5, s0 = U(rng) - .5, s1 = U(rng) - .5;
    std::vector<double> geom(5 + 3 * nv);
    double vx[8][2];
    for (int k = 0; k < nv; ++k) {
      const double a = 2 * PI_D * (k + 0.8 * U(rng)) / nv;
      vx[k][0] = size * std::cos(a) * (0.3 + U(rng));
      vx[k][1] = size * std::sin(a) * (0.3 + U(rng));
      if (degenerate == 1 && k) vx[k][0] = k & 1 ? vx[k][0] : vx[k - 1][0];     // axis-parallel edges
      if (degenerate == 2 && k == nv - 1) { vx[k][0] = vx[0][0]; vx[k][1] = vx[0][1]; }
    }
    const int i1 = (ax + 1) % 3, i2 = (i1 + 1) % 3;
    double nrm[3];
    nrm[ax] = 1; nrm[i1] = -s0; nrm[i2] = -s1;
    const double l = std::sqrt(1 + s0 * s0 + s1 * s1);
    for (double& q : nrm) q /= l;
    for (int k = 0; k < nv; ++k) {
      geom[5 + 3 * k + i1] = vx[k][0];
      geom[5 + 3 * k + i2] = vx[k][1];
      geom[5 + 3 * k + ax] = c + s0 * vx[k][0] + s1 * vx[k][1];
    }
    for (int a = 0; a < 3; ++a) geom[a] = nrm[a];
    geom[3] = nrm[0] * geom[5] + nrm[1] * geom[6] + nrm[2] * geom[7];
    geom[4] = ax;
    Prim prims[2] = {{PK_POLYGON, 0, 3, -1, 0, nv, PF_FLAT, -1}, {PK_POLYGON, 0, 2, -1, 0, nv, PF_FLAT, -1}};
    Material mat{};
    DevScene S{};
    S.prims = prims;
    S.geom = geom.data();
    S.mats = &mat;
    const LeafRec L = leaf_rec(S, 0, 0);
    if ((L.ax >= 0) != (nv == 3 || nv == 4)) return -1;
    for (int r = 0; r < nrays; ++r) {
      double p[3], u, v;
      const int k = (int)(rng() % nv), k1 = (k + 1) % nv, how = (int)(rng() % 4);
      if (how == 0) { u = (2 * U(rng) - 1) * size; v = (2 * U(rng) - 1) * size; }
      else {
        const double t = how == 1 ? 0.0 : U(rng), j = how == 3 ? 3e-6 : 1e-7;
        u = vx[k][0] + t * (vx[k1][0] - vx[k][0]) + j * (2 * U(rng) - 1);
        v = vx[k][1] + t * (vx[k1][1] - vx[k][1]) + j * (2 * U(rng) - 1);
      }
      p[i1] = u; p[i2] = v; p[ax] = c + s0 * u + s1 * v;
      V3 d = v3(2 * U(rng) - 1, 2 * U(rng) - 1, 2 * U(rng) - 1);
      if (rng() % 8 == 0) { d = v3(0, 0, 0); (ax == 0 ? d.x : ax == 1 ? d.y : d.z) = rng() & 1 ? 1 : -1; }
      normalize(d);
      const double back = 0.1 + 3 * U(rng);
      const V3 o = v3(p[0], p[1], p[2]) - d * back;
      HitRec a;
      a.t = FHUGE; a.rod = 1.0; a.prim = -1;
      if (rng() & 1) { a.t = back + 3e-6 * (2 * U(rng) - 1); a.rod = rng() & 1 ? 1.0 : -1.0; a.prim = 1; }
      HitRec b = a;
      hit_prim(S, 0, o, d, a);
      hit_leaf(S, L, 0, o, d, b);
      nhit += a.prim == 0;
      if (a.prim != b.prim || a.t != b.t || a.rod != b.rod) ++bad;
    }
  }
  *hits = nhit;
  return bad;
}

// Random boxes, their tree and its four-wide form: for random rays, the order
// in which a walk of the unrounded four-wide nodes meets the leaves (nearest
// entry first, equal entries in slot order) is the order met_before() gives
// for every pair of them, and leaf_positions() numbers the leaves left to
// right.  grid: boxes on a lattice, so that entries coincide.  Returns a bit
// mask; *pairs counts the pairs compared.
extern "C" int check_order(int n, int nrays, unsigned seed, int grid, long* pairs) {
  using namespace rg;
  std::mt19937 rng(seed);
  std::uniform_real_distribution<float> U(0.0f, 1.0f);
  std::vector<float> lo(3 * n), hi(3 * n);
  std::vector<int32_t> ids(n);
  for (int i = 0; i < n; ++i) {
    for (int a = 0; a < 3; ++a) {
      const float c = grid ? (float)(rng() % 8) : U(rng) * 10.0f, h = grid ? 0.5f : 0.05f + U(rng);
      lo[3 * i + a] = c - h;
      hi[3 * i + a] = c + h;
    }
    ids[i] = i;
  }
  std::vector<BVHNode> nodes;
  const int32_t root = build_sah_bvh(lo.data(), hi.data(), ids.data(), (uint32_t)n, nodes, 60);
  std::vector<BVH4Node> q;
  collapse_bvh4(nodes, root, q);
  const std::vector<int32_t> pos = leaf_positions(nodes, root, (size_t)n + 2);
  int bad = 0;
  if (pos[n] != -1 || pos[n + 1] != -1) bad |= 1;
  std::vector<char> seen(n, 0);
  for (int i = 0; i < n; ++i) {
    if (pos[i] < 0 || pos[i] >= n || seen[pos[i]]) bad |= 2;
    else seen[pos[i]] = 1;
  }
  DevScene S{};
  S.nodes = nodes.data();
  S.root = root;
  S.nbvh = n;
  *pairs = 0;
  for (int r = 0; r < nrays; ++r) {
    float o[3], iv[3], ot[3];
    for (int a = 0; a < 3; ++a) {
      const float d = grid && rng() % 3 == 0 ? 1e-20f : 2 * U(rng) - 1;
      o[a] = U(rng) * 12.0f - 1.0f;
      iv[a] = 1.0f / (std::fabs(d) < 1e-20f ? 1e-20f : d);
      ot[a] = o[a] * iv[a];
    }
    std::vector<int32_t> met, st{0};
    while (!st.empty()) {
      const int32_t ref = st.back();
      st.pop_back();
      if (ref < 0) { met.push_back(~ref); continue; }
      const BVH4Node& Q = q[(size_t)ref];
      std::vector<std::pair<float, int>> hits;
      for (int k = 0; k < 4; ++k) {
        if (Q.child[k] == INT32_MIN) continue;
        const float l[3] = {Q.lox[k], Q.loy[k], Q.loz[k]}, h[3] = {Q.hix[k], Q.hiy[k], Q.hiz[k]};
        float tn = -INFINITY, tf = INFINITY;
        for (int a = 0; a < 3; ++a) {
          const float t0 = std::fma(l[a], iv[a], -ot[a]), t1 = std::fma(h[a], iv[a], -ot[a]);
          tn = std::fmax(tn, std::fmin(t0, t1));
          tf = std::fmin(tf, std::fmax(t0, t1));
        }
        if (tn <= tf && tf >= 0) hits.push_back({tn, k});
      }
      std::sort(hits.begin(), hits.end());
      for (size_t k = hits.size(); k--;) st.push_back(Q.child[hits[k].second]);
    }
    for (size_t a = 0; a < met.size(); ++a)
      for (size_t b = 0; b < met.size(); ++b) {
        if (a == b) continue;
        ++*pairs;
        if (met_before(S, pos[met[a]], pos[met[b]], ot, iv) != (a < b)) bad |= 4;
      }
  }
  return bad;
}

// A ray's origin and direction as the walk holds them.
static void walk_ray(const double o[3], const double d[3], float ot[3], float iv[3]) {
  for (int a = 0; a < 3; ++a) {
    float f = (float)d[a];
    if (std::fabs(f) < 1e-20f) f = f < 0 ? -1e-20f : 1e-20f;
    iv[a] = 1.0f / f;
    ot[a] = (float)o[a] * iv[a];
  }
}

// Boxes within a scene of side `ext` about the origin, widened as a commit
// widens primitives (1e-5 + 4e-6 ext), four to a rounded node: a ray from up
// to `far` sides away through a point of an unwidened box enters that box by
// the walk's own FP32 arithmetic, also with a hit at that point already
// found.  flat: boxes without thickness in one axis, and rays along axes.
// Returns the number of rays that miss.
extern "C" long check_walk_boxes(int n, int nrays, unsigned seed, double ext, double far, int flat) {
  using namespace rg;
  std::mt19937 rng(seed);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  const double eps = 1e-5 + 4e-6 * ext;
  long bad = 0;
  for (int i = 0; i < n; ++i) {
    BVH4Node N = {};
    float* lo[3] = {N.lox, N.loy, N.loz};
    float* hi[3] = {N.hix, N.hiy, N.hiz};
    double blo[4][3], bhi[4][3];
    const double e = ext * std::pow(10.0, -4 + 4 * U(rng));
    for (int k = 0; k < 4; ++k) {
      N.child[k] = ~k;
      const int thin = flat ? (int)(rng() % 3) : -1;
      for (int a = 0; a < 3; ++a) {
        const double c = (U(rng) - 0.5) * (ext - e), h = a == thin ? 0.0 : 0.5 * e * U(rng);
        blo[k][a] = c - h;
        bhi[k][a] = c + h;
        lo[a][k] = std::nextafter((float)(blo[k][a] - eps), -INFINITY);
        hi[a][k] = std::nextafter((float)(bhi[k][a] + eps), INFINITY);
      }
    }
    const BVH4Q Q = quantize_node(N);
    for (int r = 0; r < nrays; ++r) {
      const int k = (int)(rng() & 3);
      double p[3], o[3], d[3], t = 0;
      for (int a = 0; a < 3; ++a) {
        p[a] = blo[k][a] + (bhi[k][a] - blo[k][a]) * (rng() % 4 ? U(rng) : (double)(rng() & 1));
        o[a] = (2 * U(rng) - 1) * (0.5 + far) * ext;
        if (flat && rng() % 3 == 0) o[a] = p[a];
      }
      for (int a = 0; a < 3; ++a) t += (p[a] - o[a]) * (p[a] - o[a]);
      t = std::sqrt(t);
      if (!(t > 0)) continue;
      for (int a = 0; a < 3; ++a) d[a] = (p[a] - o[a]) / t;
      float ot[3], iv[3];
      walk_ray(o, d, ot, iv);
      for (const double hit : {FHUGE, t}) {
        uint32_t key[4];
        walk_keys(Q, ot, iv, walk_limit(hit), key);
        if (key[k] == kNoEntry || (int)(key[k] & 3u) != k) ++bad;
      }
    }
  }
  return bad;
}

// Rays that are not numbers: with no axis left to bound a box, or behind a
// hit at a distance that is not a number, the walk enters nothing, as one
// that compares the slab's own ends does; with one such axis the others
// decide.  Returns a bit mask.
extern "C" int check_walk_nan(int n, unsigned seed) {
  using namespace rg;
  std::mt19937 rng(seed);
  std::uniform_real_distribution<float> U(-1.0f, 1.0f);
  const double bad_number = std::nan("");
  int bad = 0;
  for (int i = 0; i < n; ++i) {
    BVH4Node N = {};
    float* lo[3] = {N.lox, N.loy, N.loz};
    float* hi[3] = {N.hix, N.hiy, N.hiz};
    for (int k = 0; k < 4; ++k) {
      N.child[k] = ~k;
      for (int a = 0; a < 3; ++a) { lo[a][k] = U(rng); hi[a][k] = lo[a][k] + std::fabs(U(rng)); }
    }
    const BVH4Q Q = quantize_node(N);
    double o[3] = {U(rng), U(rng), U(rng)}, d[3] = {U(rng), U(rng), U(rng)};
    float ot[3], iv[3];
    uint32_t key[4], was[4];
    auto none = [&](const double* oo, const double* dd, double hit) {
      walk_ray(oo, dd, ot, iv);
      walk_keys(Q, ot, iv, walk_start(hit, ot), key);
      for (uint32_t q : key)
        if (q != kNoEntry) return false;
      return true;
    };
    const double nan3[3] = {bad_number, bad_number, bad_number};
    if (!none(o, nan3, FHUGE)) bad |= 1;
    if (!none(nan3, d, FHUGE)) bad |= 2;
    if (!none(o, d, bad_number)) bad |= 4;
    walk_ray(o, d, ot, iv);
    walk_keys(Q, ot, iv, walk_limit(bad_number), key);
    for (uint32_t q : key)
      if (q != kNoEntry) bad |= 8;
    // one axis: as if every box filled it
    const int ax = (int)(rng() % 3);
    double one[3] = {o[0], o[1], o[2]};
    one[ax] = bad_number;
    walk_ray(one, d, ot, iv);
    walk_keys(Q, ot, iv, walk_start(FHUGE, ot), key);
    for (int k = 0; k < 4; ++k) { lo[ax][k] = -1e6f; hi[ax][k] = 1e6f; }
    walk_ray(o, d, ot, iv);
    walk_keys(quantize_node(N), ot, iv, walk_start(FHUGE, ot), was);
    for (int k = 0; k < 4; ++k)
      if ((key[k] == kNoEntry) != (was[k] == kNoEntry)) bad |= 16;
  }
  return bad;
}
