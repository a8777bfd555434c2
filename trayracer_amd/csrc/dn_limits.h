// How large an image of a tensor the network's kernels can address. They read and write its
// bf16 tensors through buffer resources of one image each, whose byte offsets are 32-bit and
// unsigned; sums of offsets may wrap on the way to one that is in range.
#pragma once
#include <stdint.h>

namespace trt {

// The offset of a load that has to return zero (the convolutions' padding): past every image.
constexpr uint32_t kBufOutside = 0xfffffff0u;

// Loads of a tensor [H][W][C] bf16: every byte lies below kBufOutside.
inline bool dn_load_ok(int64_t H, int64_t W, int64_t C) { return H * W * C * 2 <= int64_t(kBufOutside); }

// Stores in tiles of `rows` rows: also the rows that the last tile has beyond the image, which
// the buffer's range drops, have offsets that do not wrap.
inline bool dn_store_ok(int64_t H, int64_t W, int64_t C, int64_t rows) {
  return (H + rows - 1) / rows * rows * W * C * 2 <= (int64_t(1) << 32);
}

}  // namespace trt
