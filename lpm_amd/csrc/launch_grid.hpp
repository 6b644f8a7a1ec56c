// Grids of launches with many blocks.  Host code with no dependencies, so that
// a test driver can include it.
#pragma once

#include <cstdint>

namespace lpm_amd {

struct GridXY {
  unsigned x, y;
};

// At least `blocks` blocks of `threads`: a launch takes fewer than 2^32
// threads in x, which 64-target blocks of 512 threads pass at 537 million
// targets; beyond, rows of equal length, a multiple of 8 as the XCD of a block
// is its index mod 8.  Kernels take blockIdx.y * gridDim.x + blockIdx.x and
// leave with a surplus index.
inline GridXY grid_xy(int64_t blocks, int threads) {
  const int64_t most = ((int64_t(1) << 32) - 1) / threads / 8 * 8;
  if (blocks <= most) return {static_cast<unsigned>(blocks), 1u};
  const int64_t rows = (blocks + most - 1) / most;
  const int64_t x = ((blocks + rows - 1) / rows + 7) / 8 * 8;
  return {static_cast<unsigned>(x), static_cast<unsigned>(rows)};
}

}  // namespace lpm_amd
