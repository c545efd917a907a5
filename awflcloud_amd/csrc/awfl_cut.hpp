// awfl_cut.hpp -- how the sweeps are cut into work-groups: rules on sizes, host
// code alone, with the timings that they rest on.
#pragma once
#include <cstdint>

namespace awfl_cut {

// ---------------------------------------------------------------------------
// sweep adjoint (k_adj_tile in awfl_adjoint.hip)
// ---------------------------------------------------------------------------
// Cells of a line, lanes of a work-group: the twelve waves that a CU holds.  The
// five kernels for longer lines, with 56 doubles (3, 2) or 76 (5, 3) of HBM per
// cell, took 1.1 to 1.2 ms for a sweep along a line of 700 cells, 160 x 40 of them,
// at (3, 2) and 1.6 ms at (5, 3); the tile takes 0.37 (x), 0.58 (y), 0.62 (z) and
// 0.53, 0.72, 0.73 ms.
constexpr int ADJ_MAX = 768;

// Lines per work-group.  Up to 256 cells, groups of at most four waves, one per
// SIMD: few idle lanes first, then whole groups of four, of which three fit a CU
// and load its SIMDs alike; never so many that CUs stay without a group.  Against
// four waves, one, two and three took 1.10, 1.06 and 1.05 times as long
// (128x128x64, z 143.8, 137.6 and 138.1 against 131.1 us; x and y by one line of
// two waves 127.9 and 139.8, by two 123.1 and 127.6), five to eight 1.09 to 1.4
// times (100x90x75, x in 500 lanes 106 against 97 us).
// Longer lines: a CU holds one group of five waves or more, whatever its size, so
// two lines share one while they fit and there are more lines than CUs (289 cells,
// 160 x 40 lines, x / y / z: 179 / 203 / 210 us against 245 / 289 / 305 one by one at
// (3, 2), 268 / 284 / 292 against 366 / 402 / 418 at (5, 3); 320 lines of 300 cells 18
// against 23 us, 224 lines 17 against 14).
inline int adj_cols(int n, int64_t lines) {
  if (n > 256) return 2 * n <= ADJ_MAX && lines > 256 ? 2 : 1;
  constexpr double slack[5] = {0, 1.10, 1.06, 1.05, 1.0};
  int best = 1;
  double cost = 1e300;
  for (int m = 1; m * n <= 256 && (m == 1 || (lines + m - 1) / m >= 256); m++) {
    const int waves = (m * n + 63) / 64;
    const double e = slack[waves] * waves / m;
    if (e < cost) {
      cost = e;
      best = m;
    }
  }
  return best;
}

}  // namespace awfl_cut
