// Check of segments.h: blocks of grids below, at and above the segment count take every item of
// every segment exactly once and come to an end. Prints "ok" or the first violation.
#include <cstddef>
#include <cstdio>
#include <vector>

#include "trt/segments.h"

using namespace trt;

int main() {
  const uint32_t n_segs = 32, threads = 4;
  const uint32_t counts[] = {0, 1, 3, 4, 5, 97, 1000};
  for (uint32_t grid = 1; grid <= 200; ++grid) {
    std::vector<std::vector<uint32_t>> taken(n_segs);
    for (uint32_t s = 0; s < n_segs; ++s) taken[s].assign(counts[s % 7], 0u);
    for (uint32_t block = 0; block < grid; ++block)
      for (uint32_t s = block % n_segs; s < n_segs; s += grid) {
        const uint32_t first = segment_place(block, n_segs) * threads, step = segment_blocks(s, grid, n_segs) * threads;
        if (step == 0) {
          std::printf("FAIL grid %u, block %u, segment %u: no progress\n", grid, block, s);
          return 1;
        }
        for (uint32_t t = 0; t < threads; ++t)
          for (uint32_t i = first + t; i < taken[s].size(); i += step) ++taken[s][i];
      }
    for (uint32_t s = 0; s < n_segs; ++s)
      for (size_t i = 0; i < taken[s].size(); ++i)
        if (taken[s][i] != 1) {
          std::printf("FAIL grid %u, segment %u: item %zu taken %u times\n", grid, s, i, taken[s][i]);
          return 1;
        }
  }
  std::printf("ok\n");
  return 0;
}
