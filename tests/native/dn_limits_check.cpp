// Check of the network kernels' address limits (dn_limits.h; host code). Over image sizes up to
// and beyond the largest: wherever the forward pass's loads and stores are in order, so are the
// backward's; offsets as the kernels form them, in wrapping 32-bit sums, are the true ones; the
// offset of a padding load lies outside of every image; and rows that a tile has beyond the
// image fall outside too. Prints "ok" and the largest square crop, or the first violation.
#include <cstddef>
#include <initializer_list>
#include <cstdio>

#include "dn_limits.h"

using namespace trt;

struct Layer {  // channels of the upsampled and the plain input, of the output; the side's divisor
  int c1, cx, cout, div;
};
static const Layer kNet[] = {{0, 16, 32, 1}, {0, 32, 32, 1}, {0, 32, 64, 2}, {0, 64, 64, 2}, {0, 64, 96, 4},
                             {0, 96, 96, 4}, {0, 96, 128, 8}, {0, 128, 128, 8}, {128, 96, 96, 4}, {0, 96, 96, 4},
                             {96, 64, 64, 2}, {0, 64, 64, 2}, {64, 32, 32, 1}, {0, 32, 32, 1}, {0, 32, 32, 1}};

static bool forward(int64_t H, int64_t W) {
  for (const Layer& l : kNet) {
    const int64_t h = H / l.div, w = W / l.div;
    if (!dn_load_ok(h, w, l.cx) || !dn_load_ok(h / 2, w / 2, l.c1)) return false;
    if (&l != &kNet[14] && !dn_store_ok(h, w, l.cout, 16)) return false;  // the last one writes fp32 by pointer
  }
  return true;
}
static bool backward(int64_t H, int64_t W) {  // input gradients are written by pointer
  for (const Layer& l : kNet) {
    const int64_t h = H / l.div, w = W / l.div;
    if (!dn_load_ok(h, w, l.cx) || !dn_load_ok(h / 2, w / 2, l.c1) || !dn_load_ok(h, w, l.cout)) return false;
  }
  return true;
}

static int fail(const char* what, int64_t H, int64_t W) {
  std::printf("FAIL %s at %lld x %lld\n", what, static_cast<long long>(H), static_cast<long long>(W));
  return 1;
}

int main() {
  size_t accepted = 0, refused = 0;
  for (int64_t W = 128; W <= 1 << 22; W = W < 9000 ? W + 128 : W * 2)
    for (int64_t H = 8; H <= 1 << 16; H += H < 64 || H > 7900 ? 8 : 504) {
      if (H > 9000 && W > 9000) break;
      const bool ok = forward(H, W);
      (ok ? accepted : refused) += 1;
      if (!ok) continue;
      if (!backward(H, W)) return fail("backward refuses what forward takes", H, W);
      const int64_t C = 32, bytes = H * W * C * 2;
      if (int64_t(kBufOutside) < bytes) return fail("padding loads lie inside the image", H, W);
      const int64_t rows = (H + 15) / 16 * 16;
      for (const int64_t y : {int64_t(0), H / 2, H - 1, rows - 1}) {
        // tile corner (first row - 1, column -1) + relative offset of row y, column W - 1
        const int64_t y0 = y / 16 * 16;
        const uint32_t corner = uint32_t(int32_t((y0 - 1) * W - 1)) * uint32_t(C) * 2u;
        const uint32_t rel = uint32_t(int32_t((y - y0 + 1) * W + W)) * uint32_t(C) * 2u;
        const int64_t at = (y * W + W - 1) * C * 2;
        if (int64_t(uint32_t(corner + rel)) != at) return fail("offset wraps", H, W);
        if (y >= H && at < bytes) return fail("a row beyond the image lies inside", H, W);
      }
    }
  if (accepted < 1000 || refused < 1000) return fail("too few sizes", int64_t(accepted), int64_t(refused));
  // as large as the fp32 input gradient of 96 channels is when its elements pass 2^31, and where bytes of a
  // 32-channel tensor pass 2^31
  if (!forward(4736, 4736) || !forward(4104, 8192)) return fail("refused", 4736, 4736);
  if (forward(8192, 8192)) return fail("accepted", 8192, 8192);
  int64_t crop = 128;
  while (forward(crop + 128, crop + 128)) crop += 128;
  std::printf("ok %lld\n", static_cast<long long>(crop));
  return 0;
}
