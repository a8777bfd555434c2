// Check of trt::slab32_ray (the per-ray terms of the slab test on 32-byte nodes): walks trees
// with directions that hit nothing, of zero or subnormal components, and counts the nodes
// they visit. The triangle test refuses them all, so they have to cost no more than the boxes
// around their origin. Prints "ok" or the first violation and exits non-zero.
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "bvh_build.h"
#include "trt/intersect.h"
#include "trt/slab32.h"

using namespace trt;

static float half_of(uint32_t h) {
  const float s = (h & 0x8000u) ? -1.f : 1.f;
  const int e = int((h >> 10) & 31u);
  if (e == 31) return s * HUGE_VALF;
  return s * (e == 0 ? std::ldexp(float(h & 1023u), -24) : std::ldexp(1024.f + float(h & 1023u), e - 25));
}

static bool enters(const uint32_t* w, V3 si, V3 oi, float tmin, float tmax) {
  const float s[3] = {si.x, si.y, si.z}, o[3] = {oi.x, oi.y, oi.z};
  float n = tmin, f = tmax;
  for (int k = 0; k < 3; ++k) {
    const float h = half_of(w[k] >> 16), ct = std::fma(half_of(w[k] & 0xffffu), s[k], o[k]);
    n = std::fmax(n, std::fma(-h, std::fabs(s[k]), ct));
    f = std::fmin(f, std::fma(h, std::fabs(s[k]), ct));
  }
  return n <= f * kBoxSlack;
}

int main() {
  const uint32_t n = 20000;
  for (const float half : {1e-3f, 1.f, 1e6f}) {
    std::mt19937 rng(11);
    std::uniform_real_distribution<float> u(-1.f, 1.f);
    std::vector<float> box(size_t(n) * 6);
    for (uint32_t i = 0; i < n; ++i)
      for (int k = 0; k < 3; ++k) {
        const float c = half * u(rng), e = 0.01f * half * std::fabs(u(rng));
        box[size_t(i) * 6 + k] = c - e;
        box[size_t(i) * 6 + 3 + k] = c + e;
      }
    const std::vector<DevNode2> dn = to_device_layout(build_binned_sah(box.data(), n, 32, 4, 2, kTravCostTriangles));
    std::vector<DevNode32> pk(dn.size());
    NodeSpace g;
    if (!pack_nodes32(dn, 0, dn.size(), g, pk.data())) return std::printf("FAIL tree refused\n"), 1;
    const V3 dirs[] = {v3(0.f), v3(-0.f, 0.f, -0.f), v3(1e-40f, 0.f, 0.f), v3(-2.9e-39f, 2.9e-39f, 1e-45f)};
    for (const V3 d : dirs)
      for (int r = 0; r < 50; ++r) {
        const V3 o = v3(half * u(rng), half * u(rng), half * u(rng));
        const float tmax = r % 2 ? 0.f : (r % 3 ? 1e30f : HUGE_VALF);  // 0: an all-zero record
        V3 si, oi;
        slab32_ray(g.org, g.step, o, d, [](float x) { return 1.f / x; }, si, oi);
        std::vector<int32_t> stack = {0};
        size_t visits = 0;
        while (!stack.empty()) {
          const int32_t node = stack.back();
          stack.pop_back();
          if (node < 0) continue;
          ++visits;
          for (int c = 0; c < 2; ++c)
            if (enters(pk[size_t(node) / 32].w + 4 * c, si, oi, 0.f, tmax)) stack.push_back(int32_t(pk[size_t(node) / 32].w[4 * c + 3]));
        }
        if (visits > dn.size() / 20) {
          std::printf("FAIL direction (%g, %g, %g), half side %g: %zu of %zu nodes visited\n", d.x, d.y, d.z, half, visits, dn.size());
          return 1;
        }
      }
    // and none of them hits a triangle, not even one around the origin
    for (const V3 d : dirs) {
      TriHit h;
      if (intersect_triangle(ray_tri_setup(v3(0.f), d), v3(-1.f, -1.f, 1e-3f), v3(1.f, -1.f, 1e-3f), v3(0.f, 2.f, -1e-3f), 0.f,
                             HUGE_VALF, h))
        return std::printf("FAIL a zero direction hits\n"), 1;
    }
  }
  std::printf("ok\n");
  return 0;
}
