// How the blocks of a grid share the segments of a segmented list: block b begins with segment
// b % n_segs. A grid of at least n_segs blocks has every segment as some blocks' first and
// only one; a smaller grid's blocks go on to every grid-th segment, each theirs alone.
#pragma once
#include "common.h"

namespace trt {

// A block's place among those of a segment, and their number.
TRT_FI uint32_t segment_place(uint32_t block, uint32_t n_segs) { return block / n_segs; }
TRT_FI uint32_t segment_blocks(uint32_t segment, uint32_t grid, uint32_t n_segs) {
  return grid < n_segs ? 1u : (grid - segment + n_segs - 1u) / n_segs;
}

}  // namespace trt
