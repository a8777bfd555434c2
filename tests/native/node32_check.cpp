// Property check of trt::pack_nodes32, the 32-byte device node layout (fp16 centre and half
// extent on the tree's grid; host code only). Prints "ok <nodes>" or the first violation and
// exits non-zero.
//   1. child references are kept (internal children as byte offsets, index x 32), and the
//      child of a leaf without triangles is never entered;
//   2. every stored box contains the exact one with its margins, and is no larger than the
//      layout's rounding explains;
//   3. rays that touch an exact child box in FP64 pass the device's float slab test
//      (ct = fma(c, si, oi), entry fma(-h, |si|, ct), exit fma(h, |si|, ct)): near and far
//      origins, short and long directions, zero and tiny components; and rays outside the
//      box's slab on an axis they are parallel to fail it;
//   4. a tree of evenly fine detail suits the layout, one of a small object in a large
//      surrounding, an infinite bound and a far too large one do not.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

#include "bvh_build.h"
#include "trt/intersect.h"

using namespace trt;

static int fail(const char* what, size_t i) {
  std::printf("FAIL %s at %zu\n", what, i);
  return 1;
}

static double half_of(uint32_t h) {
  const double s = (h & 0x8000u) ? -1.0 : 1.0;
  const int e = int((h >> 10) & 31u);
  const double m = double(h & 1023u);
  if (e == 31) return m != 0.0 ? NAN : s * HUGE_VAL;
  return s * (e == 0 ? std::ldexp(m, -24) : std::ldexp(1024.0 + m, e - 25));
}

// the device's per-ray set-up and slab test of one child (Nodes32 in kernels.hip)
struct Ray32 {
  float si[3], oi[3];
};
static Ray32 setup(const NodeSpace& g, const float* o, const float* d) {
  static int turn = 0;
  ++turn;
  Ray32 b;
  const float m = std::max(std::max(std::fabs(d[0]), std::fabs(d[1])), std::fabs(d[2])), lim = m * 0x1p-60f;
  float s_hi = 0.f, s_lo = HUGE_VALF, o_hi = 0.f, w_hi = 0.f;
  for (int k = 0; k < 3; ++k) {
    float i = 1.f / (std::fabs(d[k]) < lim ? std::copysign(lim, d[k]) : d[k]);
    i = std::nextafter(i, k == turn % 3 ? 0.f : std::copysign(HUGE_VALF, i));  // v_rcp_f32 is within an ulp
    const float w = g.org[k] - o[k];
    b.si[k] = i * g.scale;
    b.oi[k] = w * i;
    s_hi = std::max(s_hi, std::fabs(b.si[k]));
    s_lo = std::min(s_lo, std::fabs(b.si[k]));
    o_hi += std::fabs(b.oi[k]);
    w_hi += std::fabs(w);
  }
  if (!(s_lo >= 0x1p-100f && s_hi <= 0x1p100f && o_hi < 0x1p126f && w_hi < 0x1p50f * g.scale))
    for (int k = 0; k < 3; ++k) b.si[k] = 0.f, b.oi[k] = NAN;
  return b;
}
static bool slab(const uint32_t* w, const Ray32& b, float tmin, float tmax) {
  float n = tmin, f = tmax;
  for (int k = 0; k < 3; ++k) {
    const float c = float(half_of(w[k] & 0xffffu)), h = float(half_of(w[k] >> 16)), a = std::fabs(b.si[k]);
    const float ct = std::fma(c, b.si[k], b.oi[k]);
    n = std::fmax(n, std::fma(-h, a, ct));
    f = std::fmin(f, std::fma(h, a, ct));
  }
  return n <= f * kBoxSlack;
}

static std::vector<DevNode2> tree(const std::vector<float>& box) {
  return to_device_layout(build_binned_sah(box.data(), uint32_t(box.size() / 6), 32, 4, 2, kTravCostTriangles));
}

int main(int argc, char** argv) {
  const uint32_t n = argc > 1 ? uint32_t(std::atoi(argv[1])) : 8000;
  size_t nodes = 0;
  // scenes of several extents and positions: (half size, centre)
  const double scenes[][2] = {{1.0, 0.0}, {50.0, 50.0}, {1e-3, 4.0}, {3e4, -1e5}, {0x1p-30, 0.0}};
  uint64_t rays = 0, touching = 0, culled = 0, extreme = 0;
  for (const auto& sc : scenes) {
    std::mt19937 rng(7);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    std::vector<float> box(size_t(n) * 6);
    for (uint32_t i = 0; i < n; ++i)
      for (int k = 0; k < 3; ++k) {
        const double c = sc[1] + u(rng) * sc[0], e = (i + k) % 5 == 0 ? 0.0 : std::fabs(u(rng)) * sc[0] * 0.02;
        box[size_t(i) * 6 + k] = float(c - e);
        box[size_t(i) * 6 + 3 + k] = float(c + e);
      }
    const std::vector<DevNode2> dn = tree(box);
    std::vector<DevNode32> pk(dn.size());
    NodeSpace g;
    if (!pack_nodes32(dn, 0, dn.size(), g, pk.data())) return fail("evenly fine tree refused", size_t(&sc - scenes));
    nodes += dn.size();
    double R = 0.0;  // half size of the grid's tree, from the root's children
    for (int k = 0; k < 3; ++k)
      for (int c = 0; c < 2; ++c) {
        const float lo = k < 2 ? (c ? dn[0].r1 : dn[0].r0)[2 * k] : dn[0].r2[2 * c];
        const float hi = k < 2 ? (c ? dn[0].r1 : dn[0].r0)[2 * k + 1] : dn[0].r2[2 * c + 1];
        R = std::max(R, std::max(double(hi) - g.org[k], double(g.org[k]) - lo));
      }
    for (size_t i = 0; i < dn.size(); ++i) {
      const DevNode2& a = dn[i];
      for (int c = 0; c < 2; ++c) {
        const uint32_t* w = pk[i].w + 4 * c;
        const int32_t ref = a.c[c];
        if (int32_t(w[3]) != (ref >= 0 ? ref * 32 : ref)) return fail("child reference", i);
        const float* xy = c ? a.r1 : a.r0;
        const float lo[3] = {xy[0], xy[2], a.r2[2 * c]}, hi[3] = {xy[1], xy[3], a.r2[2 * c + 1]};
        double slo[3], shi[3];
        for (int k = 0; k < 3; ++k) {
          const double cs = half_of(w[k] & 0xffffu) * g.scale + g.org[k], hs = half_of(w[k] >> 16) * g.scale;
          slo[k] = cs - hs;
          shi[k] = cs + hs;
          const double need = std::max(double(hi[k]) - cs, cs - double(lo[k]));
          if (!(hs >= need * (1.0 + kHalfExtentMargin) + R * 0x1p-20)) return fail("margins", i);
          if (!(hs <= (0.5 * (double(hi[k]) - lo[k]) + R * 0x1p-11) * (1.0 + 0x1p-8))) return fail("box too large", i);
        }
        for (int r = 0; r < 16; ++r) {
          double o[3], d[3];
          const double far_by = r == 12 ? 1e3 : (r == 13 ? 1e6 : 4.0);
          const double len = r == 10 ? 1e-12 : (r == 11 ? 1e12 : 1.0);
          for (int k = 0; k < 3; ++k) {
            const double ctr = 0.5 * (double(lo[k]) + hi[k]), ext = std::max(double(hi[k]) - lo[k], 1e-6 * R);
            o[k] = ctr + u(rng) * (r >= 12 && r < 14 ? far_by * R : ext * far_by);
            const double tgt = (r & 1) ? (u(rng) > 0 ? double(hi[k]) : double(lo[k])) : ctr + 0.4 * u(rng) * (double(hi[k]) - lo[k]);
            d[k] = (tgt - o[k]) / R * len;
          }
          if (r >= 5 && r < 10) {  // parallel, or nearly, to an axis, from inside the slab or (odd) outside it
            const int k = (r + int(i)) % 3;
            d[k] = r == 7 ? -0.0 : (r == 8 ? 1e-30 : 0.0);
            o[k] = (r & 1) ? o[k] : 0.5 * (double(lo[k]) + hi[k]);
          }
          if (r >= 14) {  // from inside, just short of a face, towards it
            for (int k = 0; k < 3; ++k) {
              o[k] = lo[k] + (0.25 + 0.5 * std::fabs(u(rng))) * (double(hi[k]) - lo[k]);
              d[k] = 1e-3 * u(rng);
            }
            const int k = (r + int(i)) % 3;
            o[k] = double(hi[k]) - (double(hi[k]) - lo[k]) * 1e-6;
            d[k] = 1.0;
          }
          const float fo[3] = {float(o[0]), float(o[1]), float(o[2])}, fd[3] = {float(d[0]), float(d[1]), float(d[2])};
          double tn = 0.0, tf = 1e30;
          bool hit = true, outside = false;
          for (int k = 0; k < 3; ++k) {
            if (fd[k] == 0.f) {
              if (double(fo[k]) < lo[k] || double(fo[k]) > hi[k]) hit = false;
              if (double(fo[k]) < slo[k] - R * 0x1p-18 || double(fo[k]) > shi[k] + R * 0x1p-18) outside = true;
              continue;
            }
            double t0 = (double(lo[k]) - fo[k]) / fd[k], t1 = (double(hi[k]) - fo[k]) / fd[k];
            if (t0 > t1) std::swap(t0, t1);
            tn = std::max(tn, t0);
            tf = std::min(tf, t1);
          }
          ++rays;
          const Ray32 b = setup(g, fo, fd);
          if (std::isnan(b.oi[0])) ++extreme;
          const bool in = slab(w, b, 0.f, 1e30f);
          if (outside) {
            if (in) return fail("parallel ray outside its slab not culled", i);
            ++culled;
          }
          if (hit && tn <= tf) {
            ++touching;
            if (!in) return fail("slab test culled a box the ray touches", i);
          }
        }
      }
    }
  }
  if (touching < rays / 4 || culled < 100) return fail("too few touching or culled rays", touching);
  if (extreme != 0) return fail("an ordinary ray took the extreme path", extreme);
  // rays beyond the terms' range enter every box
  {
    const NodeSpace g{{0.f, 0.f, 0.f}, 0x1p-14f};
    const uint32_t w[3] = {0x3c003c00u, 0x3c003c00u, 0x3c003c00u};
    const float o[3] = {0.f, 0.f, 0.f}, far_o[3] = {1e30f, 0.f, 0.f}, zero[3] = {0.f, 0.f, 0.f}, tiny[3] = {1e-38f, 0.f, 0.f},
                huge[3] = {1e38f, 1.f, 1.f};
    for (const float* d : {zero, tiny, huge})
      if (!slab(w, setup(g, o, d), 0.f, 1e30f)) return fail("extreme direction culled", 0);
    if (!slab(w, setup(g, far_o, huge), 0.f, 1e30f)) return fail("extreme origin culled", 0);
  }
  // a root leaf beside its empty child
  {
    const std::vector<float> one = {1.f, 1.f, 1.f, 2.f, 2.f, 2.f};
    const std::vector<DevNode2> dn = tree(one);
    std::vector<DevNode32> pk(dn.size());
    NodeSpace g;
    if (!pack_nodes32(dn, 0, dn.size(), g, pk.data())) return fail("single box refused", 0);
    const float o[3] = {0.f, 0.f, 0.f}, d[3] = {1.f, 1.f, 1.f};
    if (!slab(pk[0].w, setup(g, o, d), 0.f, 1e30f)) return fail("single box culled", 0);
    if (slab(pk[0].w + 4, setup(g, o, d), 0.f, 1e30f)) return fail("empty child entered", 0);
  }
  // a detailed object of 1/4000 of the surrounding's size, away from its centre; unusable bounds
  {
    std::mt19937 rng(3);
    std::uniform_real_distribution<float> u(-1.f, 1.f);
    std::vector<float> box = {-1000.f, -1000.f, -1000.f, -999.f, -999.f, -999.f, 999.f, 999.f, 999.f, 1000.f, 1000.f, 1000.f};
    for (int i = 0; i < 2000; ++i) {
      float c[3];
      for (float& v : c) v = 0.25f * u(rng);
      for (int s = -1; s <= 1; s += 2)
        for (float v : c) box.push_back(600.f + v + 0.01f * float(s));
    }
    std::vector<DevNode2> dn = tree(box);
    std::vector<DevNode32> pk(dn.size());
    NodeSpace g;
    if (pack_nodes32(dn, 0, dn.size(), g, pk.data())) return fail("small object in a large surrounding accepted", 0);
    dn[0].r0[1] = HUGE_VALF;
    if (pack_nodes32(dn, 0, dn.size(), g, pk.data())) return fail("infinite bound accepted", 0);
    dn[0].r0[1] = 1e30f;
    if (pack_nodes32(dn, 0, dn.size(), g, pk.data())) return fail("bound beyond the grid accepted", 0);
  }
  std::printf("ok %zu\n", nodes);
  return 0;
}
