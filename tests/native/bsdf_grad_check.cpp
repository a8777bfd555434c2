// Error of trt::bsdf_grad and of bsdf_f on dual numbers against 64-bit derivatives of the
// same formulas (complex step in std::complex<double>, from the float inputs). Prints, per
// parameter, both relative errors in 2-norm over random materials and directions, and the
// largest error of each relative to the derivative's size in its material, then "ok" when
// bsdf_grad is no further off.
#include <cmath>
#include <complex>
#include <cstdio>
#include <random>

#include "trt/bsdf.h"

using namespace trt;
typedef std::complex<double> C;

static C cmaxd(C a, double b) { return a.real() > b ? a : C(b, 0.0); }
static double schlick(double c) { const double m = std::min(1.0, std::max(0.0, 1.0 - c)); return m * m * m * m * m; }

// f of the models' formulas, theta = base r, g, b, roughness, metallic
static void f64(const BsdfParams<float>& p, const C th[5], V3 wo, V3 wi, C out[3]) {
  if (p.model == kModelLambert) {
    for (int c = 0; c < 3; ++c) out[c] = th[c] / M_PI;
    return;
  }
  const double o[3] = {wo.x, wo.y, wo.z}, i[3] = {wi.x, wi.y, wi.z};
  double h[3], n = 0.0;
  for (int k = 0; k < 3; ++k) { h[k] = o[k] + i[k]; n += h[k] * h[k]; }
  for (double& v : h) v /= std::sqrt(n);
  const double cl = i[2], cv = o[2], cd = i[0] * h[0] + i[1] * h[1] + i[2] * h[2];
  const double FL = schlick(cl), FV = schlick(cv), FH = schlick(cd);
  const C r = th[3], m = th[4], lum = 0.2126729 * th[0] + 0.7151522 * th[1] + 0.0721750 * th[2];
  const C fd90 = 0.5 + 2.0 * r * cd * cd;
  C dw = (1.0 + (fd90 - 1.0) * FL) * (1.0 + (fd90 - 1.0) * FV);
  if (p.subsurface > 0.f) {
    const C fs = r * cd * cd;
    const C fss = (1.0 + (fs - 1.0) * FL) * (1.0 + (fs - 1.0) * FV);
    dw = (1.0 - double(p.subsurface)) * dw + double(p.subsurface) * 1.25 * (fss * (1.0 / (cl + cv) - 0.5) + 0.5);
  }
  const double asp = std::sqrt(1.0 - 0.9 * double(p.anisotropic));
  const C ax = cmaxd(r * r / asp, 1e-3), ay = cmaxd(r * r * asp, 1e-3);
  const C t = h[0] * h[0] / (ax * ax) + h[1] * h[1] / (ay * ay) + h[2] * h[2];
  const C D = 1.0 / (M_PI * ax * ay * t * t);
  auto lam = [&](const double* w) { return (std::sqrt(1.0 + (ax * ax * w[0] * w[0] + ay * ay * w[1] * w[1]) / (w[2] * w[2])) - 1.0) * 0.5; };
  const C spec = D / (1.0 + lam(o) + lam(i)) / (4.0 * cl * cv);
  for (int c = 0; c < 3; ++c) {
    const C tint = lum.real() > 0.0 ? th[c] / lum : C(1.0, 0.0);
    out[c] = th[c] * dw / M_PI * (1.0 - m);
    if (p.sheen > 0.f) out[c] += ((1.0 - double(p.sheen_tint)) + double(p.sheen_tint) * tint) * (1.0 - m) * FH * double(p.sheen);
    const C c0 = m * th[c] + (1.0 - m) * (0.08 * double(p.specular) * ((1.0 - double(p.specular_tint)) + double(p.specular_tint) * tint));
    out[c] += (c0 + (1.0 - c0) * FH) * spec;
  }
}

int main() {
  std::mt19937 rng(17);
  std::uniform_real_distribution<float> u(0.f, 1.f);
  auto dir = [&](float lo) {
    const float z = lo + (1.f - lo) * u(rng), a = 6.2831853f * u(rng), s = std::sqrt(std::max(0.f, 1.f - z * z));
    return v3(s * std::cos(a), s * std::sin(a), z);
  };
  double err[2][5] = {}, ref[5] = {}, worst[2][5] = {};
  for (int n = 0; n < 400000; ++n) {
    BsdfParams<float> p;
    p.base = t3(u(rng), u(rng), u(rng));
    p.roughness = 0.05f + 0.95f * u(rng);
    p.metallic = n % 5 == 0 ? 0.f : (n % 5 == 1 ? 1.f : u(rng));
    p.specular = u(rng);
    const bool extra = n % 2 == 0;
    p.specular_tint = extra ? u(rng) : 0.f;
    p.sheen = extra ? u(rng) : 0.f;
    p.sheen_tint = u(rng);
    p.clearcoat = extra ? u(rng) : 0.f;
    p.clearcoat_gloss = u(rng);
    p.subsurface = extra ? u(rng) : 0.f;
    p.anisotropic = extra ? 0.9f * u(rng) : 0.f;
    p.model = n % 97 == 0 ? kModelLambert : kModelDisney;
    if (n % 101 == 0) p.base = t3(0.f, 0.f, 0.f);
    const V3 wo = dir(0.05f);
    const V3 wi = n % 3 ? dir(0.05f) : normalize(v3(-wo.x + 0.1f * (u(rng) - 0.5f), -wo.y + 0.1f * (u(rng) - 0.5f), wo.z));
    float g[5][3];
    bsdf_grad(p, wo, wi, g);
    BsdfParams<Dual<5>> d;
    d.base = t3(dvar<5>(p.base.x, 0), dvar<5>(p.base.y, 1), dvar<5>(p.base.z, 2));
    d.roughness = dvar<5>(p.roughness, 3);
    d.metallic = dvar<5>(p.metallic, 4);
    d.specular = p.specular; d.specular_tint = p.specular_tint; d.sheen = p.sheen; d.sheen_tint = p.sheen_tint;
    d.clearcoat = p.clearcoat; d.clearcoat_gloss = p.clearcoat_gloss; d.subsurface = p.subsurface;
    d.anisotropic = p.anisotropic; d.model = p.model;
    const T3<Dual<5>> fd = bsdf_f(d, wo, wi);
    for (int k = 0; k < 5; ++k) {
      C th[5] = {p.base.x, p.base.y, p.base.z, p.roughness, p.metallic}, out[3];
      th[k] += C(0.0, 1e-100);
      f64(p, th, wo, wi, out);
      double scale = 0.0;
      for (int c = 0; c < 3; ++c) scale = std::max(scale, std::fabs(out[c].imag() * 1e100));
      const double dual[3] = {fd.x.d[k], fd.y.d[k], fd.z.d[k]};
      for (int c = 0; c < 3; ++c) {
        const double x = out[c].imag() * 1e100, e0 = dual[c] - x, e1 = double(g[k][c]) - x;
        ref[k] += x * x;
        err[0][k] += e0 * e0;
        err[1][k] += e1 * e1;
        if (scale > 1e-3) {
          worst[0][k] = std::max(worst[0][k], std::fabs(e0) / scale);
          worst[1][k] = std::max(worst[1][k], std::fabs(e1) / scale);
        }
      }
    }
  }
  bool ok = true;
  for (int k = 0; k < 5; ++k) {
    const double a = std::sqrt(err[0][k] / ref[k]), b = std::sqrt(err[1][k] / ref[k]);
    std::printf("theta %d: relative error dual %.2e, bsdf_grad %.2e; worst %.2e, %.2e\n", k, a, b, worst[0][k], worst[1][k]);
    ok = ok && b <= 1.05 * a + 1e-7;
  }
  std::printf(ok ? "ok\n" : "FAIL\n");
  return ok ? 0 : 1;
}
