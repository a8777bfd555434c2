// Error of trt::bsdf_grad and of bsdf_f on dual numbers against 64-bit derivatives at the
// edges: roughness down to zero, where the GGX alphas are clamped, and directions down to a
// cosine of 1e-4. Per parameter and edge:
//   bsdf_grad's mean error relative to the derivative's size in its material may be 1.1 times
// the dual numbers' (means of 400000 values: what is left is the order of the operations);
//   its largest error is below 64 ulp of the magnitudes that the derivative is added up from,
// each a product of fewer than 32 rounded factors, squares among them: (1 + 1 / (cl + cv)) for the
// diffuse and subsurface terms, q (1 + 4 / roughness) for the specular ones (|d ln alpha| is 2 /
// roughness per axis, none where it is clamped, below a roughness of 0.017), by (1 + 1 / luminance)
// for the tint.
// Prints the errors, then "ok".
#define main bsdf_grad_check_main  // f64 and its helpers
#include "bsdf_grad_check.cpp"
#undef main

int main() {
  std::mt19937 rng(29);
  std::uniform_real_distribution<float> u(0.f, 1.f);
  auto dir = [&](float z) {
    const float a = 6.2831853f * u(rng), s = std::sqrt(std::max(0.f, 1.f - z * z));
    return v3(s * std::cos(a), s * std::sin(a), z);
  };
  bool ok = true;
  for (int edge = 0; edge < 4; ++edge) {  // clamped alphas; wo, wi and both grazing
    double mean[2][5] = {}, worst[2][5] = {};
    size_t terms[5] = {};
    size_t clamped = 0, grazing = 0;
    for (int n = 0; n < 200000; ++n) {
      BsdfParams<float> p;
      p.base = t3(u(rng), u(rng), u(rng));
      p.roughness = edge == 0 ? 0.06f * u(rng) : u(rng);
      if (edge == 0 && n % 50 == 0) p.roughness = 0.f;
      p.metallic = n % 5 == 0 ? 0.f : (n % 5 == 1 ? 1.f : u(rng));
      p.specular = u(rng);
      p.specular_tint = u(rng);
      p.sheen = u(rng);
      p.sheen_tint = u(rng);
      p.clearcoat = u(rng);
      p.clearcoat_gloss = u(rng);
      p.subsurface = n % 2 ? u(rng) : 0.f;
      p.anisotropic = n % 3 ? 0.9f * u(rng) : 0.f;
      p.model = kModelDisney;
      const double asp = std::sqrt(1.0 - 0.9 * double(p.anisotropic)), r2 = double(p.roughness) * p.roughness;
      // next to where an alpha meets its clamp the two sides may fall on either side of it
      if (std::fabs(r2 / asp - 1e-3) < 1e-6 || std::fabs(r2 * asp - 1e-3) < 1e-6) continue;
      clamped += r2 / asp < 1e-3 && r2 * asp < 1e-3;
      const float z[2] = {std::pow(10.f, -4.f + 3.f * u(rng)), std::pow(10.f, -4.f + 3.f * u(rng))};
      const V3 wo = dir(edge == 1 || edge == 3 ? z[0] : 0.05f + 0.95f * u(rng));
      V3 wi = dir(edge >= 2 ? z[1] : 0.05f + 0.95f * u(rng));
      if (n % 3 == 0) wi = normalize(v3(-wo.x + 0.1f * (u(rng) - 0.5f), -wo.y + 0.1f * (u(rng) - 0.5f), wi.z));  // near the mirror direction
      grazing += wo.z < 0.05f || wi.z < 0.05f;
      const double o[3] = {wo.x, wo.y, wo.z}, in[3] = {wi.x, wi.y, wi.z};
      double h[3], norm = 0.0;
      for (int k = 0; k < 3; ++k) {
        h[k] = o[k] + in[k];
        norm += h[k] * h[k];
      }
      const double ax = std::max(r2 / asp, 1e-3), ay = std::max(r2 * asp, 1e-3);
      const double t = (h[0] * h[0] / (ax * ax) + h[1] * h[1] / (ay * ay) + h[2] * h[2]) / norm;
      const double q = 1.0 / (M_PI * ax * ay * t * t * 4.0 * o[2] * in[2]);  // G <= 1
      const double lum = 0.2126729 * p.base.x + 0.7151522 * p.base.y + 0.0721750 * p.base.z;
      const double magnitude = (1.0 + 1.0 / (o[2] + in[2]) + q * (1.0 + 4.0 / std::max(double(p.roughness), 0.017))) * (1.0 + 1.0 / lum);
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
          if (!std::isfinite(g[k][c])) {
            std::printf("FAIL theta %d: not finite (roughness %g, cosines %g, %g)\n", k, p.roughness, wo.z, wi.z);
            return 1;
          }
          worst[0][k] = std::max(worst[0][k], std::fabs(e0) / (magnitude * 0x1p-24));
          worst[1][k] = std::max(worst[1][k], std::fabs(e1) / (magnitude * 0x1p-24));
          if (scale <= 1e-3) continue;
          mean[0][k] += std::fabs(e0) / scale;
          mean[1][k] += std::fabs(e1) / scale;
          ++terms[k];
        }
      }
    }
    if (edge == 0 ? clamped < 10000 : grazing < 50000) {
      std::printf("FAIL edge %d is hardly met\n", edge);
      return 1;
    }
    for (int k = 0; k < 5; ++k) {
      const double a = mean[0][k] / double(terms[k]), b = mean[1][k] / double(terms[k]);
      const bool fine = terms[k] > 10000 && b <= 1.1 * a && worst[1][k] <= 64.0;
      std::printf("edge %d theta %d: mean relative error dual %.2e, bsdf_grad %.2e; worst, in ulp of its terms, %.1f, %.1f%s\n", edge, k, a, b,
                  worst[0][k], worst[1][k], fine ? "" : " FAIL");
      ok = ok && fine;
    }
  }
  std::printf(ok ? "ok\n" : "FAIL\n");
  return ok ? 0 : 1;
}
