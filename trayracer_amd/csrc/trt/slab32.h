// Per-ray terms of the slab test on 32-byte nodes (DevNode32), shared by the traversal and
// its host checks; the reciprocal is the caller's (v_rcp_f32 on the device).
#pragma once
#include "common.h"

namespace trt {

// With world = org + step * c on the tree's grid, a plane at c on an axis is reached at
// fma(c, si, oi): si = step / d, oi = (org - o) / d.
//   A direction component below 2^-60 of the largest takes that magnitude (v_rcp_f32's ulp
// scales all of the axis's distances alike), which moves no ray by more than the boxes'
// margins.
//   Rays so extreme that a term could overflow (in range: |si| in [2^-100, 2^100], |oi| < 2^126,
// |org - o| < 2^50 step, 2^36 times the tree's half size, all finite) take every box (NaN, which
// the axes' max and min ignore): slow and still exact.
//   Except that a direction of at most 2^-128 on every axis hits no triangle (the triangle
// test's 1 / d is infinite there and its distance NaN): it is walked as one of components 2^-60,
// which enters the boxes around the origin only. (256 such rays, as a caller pads a batch with,
// took 81 ms through every box of a 20000-triangle soup.)
template <class Rcp>
TRT_FI void slab32_ray(const float org[3], const float step[3], V3 o, V3 d, Rcp rcp, V3& si, V3& oi) {
  const float size = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(d.x), __builtin_fabsf(d.y)), __builtin_fabsf(d.z));
  const float lim = size * 0x1p-60f;
  const float ix = rcp(__builtin_fabsf(d.x) < lim ? __builtin_copysignf(lim, d.x) : d.x);
  const float iy = rcp(__builtin_fabsf(d.y) < lim ? __builtin_copysignf(lim, d.y) : d.y);
  const float iz = rcp(__builtin_fabsf(d.z) < lim ? __builtin_copysignf(lim, d.z) : d.z);
  const V3 w = v3(org[0] - o.x, org[1] - o.y, org[2] - o.z);
  si = v3(ix * step[0], iy * step[1], iz * step[2]);
  oi = v3(w.x * ix, w.y * iy, w.z * iz);
  const float s_hi = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(si.x), __builtin_fabsf(si.y)), __builtin_fabsf(si.z));
  const float s_lo = __builtin_fminf(__builtin_fminf(__builtin_fabsf(si.x), __builtin_fabsf(si.y)), __builtin_fabsf(si.z));
  const float o_hi = __builtin_fabsf(oi.x) + __builtin_fabsf(oi.y) + __builtin_fabsf(oi.z);
  const float w_hi = __builtin_fabsf(w.x) + __builtin_fabsf(w.y) + __builtin_fabsf(w.z);
  if (!(s_lo >= 0x1p-100f && s_hi <= 0x1p100f && o_hi < 0x1p126f && w_hi * 0x1p-50f < step[0])) {
    const float far = size <= 0x1p-128f ? 0x1p60f : 0.f;
    si = v3(far * step[0], far * step[1], far * step[2]);
    oi = far > 0.f ? v3(w.x * far, w.y * far, w.z * far) : v3(__builtin_nanf(""));
  }
}

}  // namespace trt
