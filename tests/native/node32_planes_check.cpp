// Check of trt::pack_nodes32 on trees with finely divided axis-aligned surfaces. Prints "ok" or
// the first violation and exits non-zero.
//   1. the flat boxes of the two most divided planes of an axis stay thin, of the most divided one
//      where the grid has one step, whatever the planes' heights, and every stored box contains
//      the exact one;
//   2. rays that touch an exact box in FP64 pass the float slab test of the traversal, grazing
//      rays among them;
//   3. a tree with many flat boxes in further planes, off the grid, is refused, one with few is not.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "bvh_build.h"
#include "trt/intersect.h"
#include "trt/slab32.h"

using namespace trt;

static int fail(const char* what, size_t i) {
  std::printf("FAIL %s at %zu\n", what, i);
  return 1;
}

static double half_of(uint32_t h) {
  const double s = (h & 0x8000u) ? -1.0 : 1.0;
  const int e = int((h >> 10) & 31u);
  if (e == 31) return s * HUGE_VAL;
  return s * (e == 0 ? std::ldexp(double(h & 1023u), -24) : std::ldexp(1024.0 + double(h & 1023u), e - 25));
}

// the slab test of Nodes32 in kernels.hip
static bool enters(const uint32_t* w, V3 si, V3 oi, float tmin, float tmax) {
  const float s[3] = {si.x, si.y, si.z}, o[3] = {oi.x, oi.y, oi.z};
  float n = tmin, f = tmax;
  for (int k = 0; k < 3; ++k) {
    const float h = float(half_of(w[k] >> 16)), ct = std::fma(float(half_of(w[k] & 0xffffu)), s[k], o[k]);
    n = std::fmax(n, std::fma(-h, std::fabs(s[k]), ct));
    f = std::fmin(f, std::fma(h, std::fabs(s[k]), ct));
  }
  return n <= f * kBoxSlack;
}

// n x n cells of a square of half side `half` at height y on `axis`
static void plane(std::vector<float>& box, int axis, float y, float half, int n) {
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j) {
      float lo[3], hi[3];
      const int u = (axis + 1) % 3, v = (axis + 2) % 3;
      lo[axis] = hi[axis] = y;
      lo[u] = half * (2.f * float(i) / float(n) - 1.f);
      hi[u] = half * (2.f * float(i + 1) / float(n) - 1.f);
      lo[v] = half * (2.f * float(j) / float(n) - 1.f);
      hi[v] = half * (2.f * float(j + 1) / float(n) - 1.f);
      box.insert(box.end(), lo, lo + 3);
      box.insert(box.end(), hi, hi + 3);
    }
}

static std::vector<DevNode2> tree(const std::vector<float>& box) {
  return to_device_layout(build_binned_sah(box.data(), uint32_t(box.size() / 6), 32, 4, 4, kTravCostTriangles));
}

int main() {
  std::mt19937 rng(5);
  std::uniform_real_distribution<float> u(-1.f, 1.f);
  auto detail = [&](std::vector<float>& box, float size) {  // an object above the lower plane
    for (int i = 0; i < 4000; ++i) {
      float lo[3], hi[3];
      for (int k = 0; k < 3; ++k) {
        const float c = size * u(rng), e = 0.05f * size * std::fabs(u(rng));
        lo[k] = c - e;
        hi[k] = c + e;
      }
      box.insert(box.end(), lo, lo + 3);
      box.insert(box.end(), hi, hi + 3);
    }
  };
  // (half side, heights): a floor, a hall, a hall about its centre, far from the origin
  const float scenes[][3] = {{5.f, -1.00317f, -1.00317f}, {50.f, -1.00317f, 3.7713f}, {3.f, -3.01f, 2.97f}, {700.f, -1.0003f, 44.123f}};
  for (int turn = 0; turn < 6; ++turn)
    for (const auto& sc : scenes) {
      const int axis = turn % 3;
      const bool stretch = turn < 3;
      std::vector<float> box;
      detail(box, std::min(1.f + sc[0] * 0.01f, 8.f));
      plane(box, axis, sc[1], sc[0], 100);
      if (sc[2] != sc[1]) plane(box, axis, sc[2], sc[0], 90);
      const std::vector<DevNode2> dn = tree(box);
      std::vector<DevNode32> pk(dn.size());
      NodeSpace g;
      if (!pack_nodes32(dn, 0, dn.size(), g, pk.data(), 4, stretch)) return fail("planes refused", size_t(axis));
      for (const float step : g.step)
        if (!stretch && step != g.scale) return fail("more than one step", size_t(axis));
      double Rk = 0.0;  // the tree's half side on the axis
      {
        double lo = HUGE_VAL, hi = -HUGE_VAL;
        for (size_t i = 0; i < box.size(); i += 6) {
          lo = std::min(lo, double(box[i + size_t(axis)]));
          hi = std::max(hi, double(box[i + 3 + size_t(axis)]));
        }
        Rk = 0.5 * (hi - lo);
      }
      size_t touching = 0, rays = 0;
      for (size_t i = 0; i < dn.size(); ++i)
        for (int c = 0; c < 2; ++c) {
          const uint32_t* w = pk[i].w + 4 * c;
          const float* xy = c ? dn[i].r1 : dn[i].r0;
          const float lo[3] = {xy[0], xy[2], dn[i].r2[2 * c]}, hi[3] = {xy[1], xy[3], dn[i].r2[2 * c + 1]};
          for (int k = 0; k < 3; ++k) {
            const double cs = half_of(w[k] & 0xffffu) * g.step[k] + g.org[k], hs = half_of(w[k] >> 16) * g.step[k];
            if (!(cs - hs <= lo[k] && cs + hs >= hi[k])) return fail("box not contained", i);
            if (k == axis && lo[k] == hi[k] && (lo[k] == sc[1] || (stretch && lo[k] == sc[2])) && !(hs <= Rk * 0x1p-18))
              return fail("thick box of a plane", i);
          }
          for (int r = 0; r < 8; ++r) {
            double o[3], d[3];
            for (int k = 0; k < 3; ++k) {
              o[k] = 0.5 * (double(lo[k]) + hi[k]) + u(rng) * (r < 4 ? sc[0] : 4.0 * (double(hi[k]) - lo[k]) + 1e-4 * sc[0]);
              d[k] = lo[k] + (0.5 + 0.5 * u(rng)) * (double(hi[k]) - lo[k]) - o[k];
            }
            if (r & 1) {  // in the plane, or grazing it
              o[axis] = lo[axis];
              d[axis] = (r & 2) ? 1e-6 * u(rng) * sc[0] : 0.0;
            }
            const float fo[3] = {float(o[0]), float(o[1]), float(o[2])}, fd[3] = {float(d[0]), float(d[1]), float(d[2])};
            double tn = 0.0, tf = 1e30;
            bool hit = fd[0] != 0.f || fd[1] != 0.f || fd[2] != 0.f;
            for (int k = 0; k < 3; ++k) {
              if (fd[k] == 0.f) {
                hit = hit && double(fo[k]) >= lo[k] && double(fo[k]) <= hi[k];
                continue;
              }
              double t0 = (double(lo[k]) - fo[k]) / fd[k], t1 = (double(hi[k]) - fo[k]) / fd[k];
              if (t0 > t1) std::swap(t0, t1);
              tn = std::max(tn, t0);
              tf = std::min(tf, t1);
            }
            ++rays;
            if (!hit || !(tn <= tf)) continue;
            ++touching;
            for (int ulp = -1; ulp <= 1; ++ulp) {  // v_rcp_f32 is within an ulp
              V3 si, oi;
              slab32_ray(g.org, g.step, v3(fo[0], fo[1], fo[2]), v3(fd[0], fd[1], fd[2]),
                         [ulp](float x) { return ulp ? std::nextafter(1.f / x, ulp * HUGE_VALF) : 1.f / x; }, si, oi);
              if (!enters(w, si, oi, 0.f, 1e30f)) return fail("slab test culled a box the ray touches", i);
            }
          }
        }
      if (touching < rays / 8) return fail("too few touching rays", touching);
    }
  // five planes of which two can be on the grid
  for (const int n : {20, 400}) {
    std::vector<float> box;
    detail(box, 1.f);
    for (int i = 0; i < 5; ++i) plane(box, 1, -2.f + 0.8f * float(i) + 0.0137f * float(i * i), 2.f, n);
    const std::vector<DevNode2> dn = tree(box);
    std::vector<DevNode32> pk(dn.size());
    NodeSpace g;
    if (pack_nodes32(dn, 0, dn.size(), g, pk.data(), 4) != (n == 20)) return fail(n == 20 ? "few boxes refused" : "thick planes accepted", size_t(n));
  }
  std::printf("ok\n");
  return 0;
}
