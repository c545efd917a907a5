// awfl_cut.hpp -- how the sweeps are cut into work-groups: rules on sizes, host
// code alone, with the timings that they rest on.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>

namespace awfl_cut {

// ---------------------------------------------------------------------------
// tile sweeps (awfl_tile.hpp) and column walkers
// ---------------------------------------------------------------------------
// How a sweep is cut: lines per work-group, rows (lanes along a line),
// segments per line and their length.
struct TilePlan {
  int cols, rows, nseg, seglen;
};

constexpr int MAX_THREADS = 1024;

// LDS elements of a work-group: staged cells and face slots
inline size_t lds_elems(const TilePlan& p, int hs) { return (size_t)5 * p.cols * (2 * p.rows + 2 * hs + 1); }

// TX choices of y and z tiles
constexpr int TX_OF[3] = {4, 8, 16};

// Rates of a sweep's kernels for the models below, in microseconds: a tile's
// wave (one cell a lane), the factor of 4-line tiles (short runs of memory),
// the factors of work-groups of 5 to 8 waves (how they pack on a CU), and the
// column walker's step with x waves on a SIMD, max(walk_least, walk x + walk_0); x
// up to whole_x counts as the next whole number (a SIMD's last round costs as much
// with one wave on a few of them as on all).
struct Rates {
  double tile, narrow, pack[4];
  double walk, walk_0, walk_least;
  double whole_x;
};

// FP64.  The (5, 3) rates are fitted to sweeps of 64x64x32 to 512x512x256 cells,
// every cut timed: best tiles 9 us at 64x64x32 (y and z; the walkers 55), 43 and 45
// at 128x128x64 (57 and 62), 84 and 92 at 160x160x80 (124 and 131), 147 and 161 at
// 192x192x96 (160 and 167), 228 and 271 at 96x300x200 (319 and 364), 340 and 393 at
// 256x256x128 (330 and 340).  The z kernel has 112 registers, four waves per SIMD,
// which work-groups of five to eight waves fill badly.  At (3, 2) the walkers are
// ahead earlier, in z above all, which rates of their own say (the tile's factors, and
// so its cut, are (5, 3)'s).  Fitted to 860 grids of 0.02 to 12 million cells, both
// forms timed: z tile and walker 355 and 284 us at 1000x160x64, 230 and 183 at
// 600x160x64, 157 and 116 at 1101x616x6, 34 and 42 at 128x128x64, 92 and 106 at
// 512x100x60.  They choose the slower form by more than 2% at 14 (y) and 17 (z) of the
// grids; (5, 3)'s did at 31 and 68, by up to 31%.
inline const Rates& rates_f64(int dir, int ord) {
  static constexpr Rates xy{2.55, 1.03, {1.15, 1.18, 1.12, 1.07}, 2.3, 0.8, 3.2, 0.0};
  static constexpr Rates z{2.6, 1.03, {1.4, 1.33, 1.2, 1.15}, 2.35, 0.9, 3.4, 0.0};
  static constexpr Rates y3{2.42, 1.03, {1.15, 1.18, 1.12, 1.07}, 1.77, 1.25, 3.24, 8.0};
  static constexpr Rates z3{1.51, 1.03, {1.4, 1.33, 1.2, 1.15}, 1.08, 0.62, 2.51, 8.0};
  if (ord == 3) return dir < 2 ? y3 : z3;
  return dir < 2 ? xy : z;
}

// FP32.  Fitted at (5, 3) to: tiles 8 us at 64x64x32 (y and z; the walkers 46 and
// 43), 25 at 120x100x60 (51 and 56), 33 at 128x128x64 (48), 108 and 112-128 at
// 192x192x96 (103 and 104), 234 and 260 at 256x256x128 (230 and 218), 1947 and 1999 at
// 512x512x256 (1545 and 1609).  At (3, 2) to 860 grids as above:
// z 162 (tile) and 140 (walker) at 600x160x64, 102 and 78 at 192x192x96, 24 and 35 at
// 128x128x64, 94 and 80 at 518x102x66; y 59 and 55 at 512x100x60, 102 and 78 at
// 192x192x96, 156 and 185 at 96x300x200.  Slower by more than 2% at 16 (y) and 20 (z) of
// them; with (5, 3)'s 27 and 33, by up to 45%.
inline const Rates& rates_f32(int dir, int ord) {
  static constexpr Rates yz{1.75, 1.2, {1.15, 1.18, 1.12, 1.07}, 1.4, 1.0, 2.7, 0.0};
  static constexpr Rates y3{1.60, 1.2, {1.15, 1.18, 1.12, 1.07}, 0.92, 1.79, 0.87, 0.0};
  static constexpr Rates z3{1.35, 1.2, {1.15, 1.18, 1.12, 1.07}, 0.89, 1.06, 3.08, 0.0};
  return ord != 3 ? yz : dir == 1 ? y3 : z3;
}

struct TileCut {
  int tx;                     // index into TX_OF (y, z)
  TilePlan p;
  int threads;
  double us;                  // modelled time
};

// Cut of a sweep of n-cell lines, nline of them side by side in each of `other`
// rows: the one of least modelled time, a tile's latency (some 5 us from its
// loads to its stores) plus the issue time of the waves that a SIMD gets (256
// CUs of four SIMDs; small grids in whole rounds).  An idle lane costs three
// quarters of a busy one.  `whole`: x lines that are updated in place, which a
// work-group must hold whole.  Other x lines of more than 512 cells run in
// segments: a group of 9 to 16 waves leaves a CU's places empty and its barriers
// uncovered (160 x 64 lines at (5, 3), whole against the best segments: 513 cells
// 336 and 219 us, 640 356 and 273, 800 435 and 328, 1024 456 and 427; at (3, 2) 249
// and 158, 269 and 194, 328 and 234, 345 and 311).  Short x lines fill a wave where
// there are as many (8x91x9, one line against 8 to a group: 11.1 and 6.0 us at (5, 3),
// 8.1 and 5.3 at (3, 2)).
inline TileCut tile_cut(int dir, int n, int nline, int other, bool per, const Rates& rate, bool whole = false) {
  TileCut best{};
  best.us = 1e300;
  auto consider = [&](int tx, int cols, int nseg, int limit) {
    const int seglen = (n + nseg - 1) / nseg;
    if ((n + seglen - 1) / seglen != nseg) return;
    const int rows = nseg == 1 ? n : !per && nseg == 2 ? seglen + 1 : seglen + 2;
    if (rows * cols > limit) return;
    const int waves = (rows * cols + 63) / 64;
    const double wgs = (double)nseg * ((nline + cols - 1) / cols) * other;
    const double rounds = wgs <= 1024 ? (double)(((int64_t)wgs + 255) / 256) : wgs / 256;
    const double eq = (0.75 * waves + 0.25 * rows * cols / 64.0) * (waves > 4 ? rate.pack[std::min(waves, 8) - 5] : 1.0) *
                      (dir > 0 && cols == 4 ? rate.narrow : 1.0);
    const double us = 5.0 + rate.tile * std::max(rounds * eq / 4, (double)((waves + 3) / 4));
    if (us < best.us) best = TileCut{tx, TilePlan{cols, rows, nseg, seglen}, waves * 64, us};
  };
  if (dir == 0) {
    if (whole || n <= 512)
      for (int cols = std::max(1, std::min(nline, 64 / n)); cols <= std::max(1, std::min(nline, 512 / n)); cols++)
        consider(0, cols, 1, MAX_THREADS);
    else
      for (int nseg = 2; nseg <= n / 64; nseg++) consider(0, 1, nseg, 512);
  } else {
    for (int x = 0; x < 3; x++)
      for (int nseg = 1; nseg <= std::max(1, n / 14); nseg++) consider(x, TX_OF[x], nseg, 512);
  }
  return best;
}

// Cut of a column-walker sweep (a lane walks a segment of its column; y and z):
// segments of at most 32 cells, and shorter (down to 16) where that is needed
// for ~4 waves per SIMD.  Modelled time: every wave reconstructs two cells more
// than its segment has.
struct WalkCut {
  int bx, nseg, seglen;
  double us;
};
inline WalkCut walk_cut(int n, int nx, int other, const Rates& rate) {
  WalkCut w{};
  w.bx = (nx + 63) / 64;
  const int64_t layer = (int64_t)w.bx * other;
  const int nseg = (int)std::max<int64_t>(1, std::min<int64_t>(std::max<int64_t>((4096 + layer - 1) / layer, (n + 31) / 32),
                                                               std::max(1, n / 16)));
  w.seglen = (n + nseg - 1) / nseg;
  w.nseg = (n + w.seglen - 1) / w.seglen;
  double x = (double)(layer * w.nseg) / 1024.0;
  if (x <= rate.whole_x) x = std::ceil(x);
  w.us = (w.seglen + 2) * std::max(rate.walk * x + rate.walk_0, rate.walk_least);
  return w;
}

// Groups of two waves with m lines each, of which some of the 256 CUs get a second
// one: the two share a SIMD, which four waves alone do not.  The WENO3 adjoint along 36
// cells of 636 lines takes 13.4 us by twos (318 groups) and 10.9 one by one, three
// tracers along 63 cells of 770 lines 11.2 and 9.7.  Grids on which groups of one wave
// leave a SIMD one at most do without.
inline bool pairs_collide(int n, int m, int64_t lines) {
  const int64_t groups = (lines + m - 1) / m;
  return n <= 64 && m * n > 64 && m * n <= 128 && groups > 256 && groups <= 512 && lines <= 1024 * (64 / n);
}

// ---------------------------------------------------------------------------
// tracer tiles and walkers (k_tile_tr, k_walk_tr in awfl_tracers.hip)
// ---------------------------------------------------------------------------
constexpr int TT_MAX = 1024;    // lanes of a work-group

constexpr int tt_stride(int ntr) { return ntr | 1; }
inline size_t tt_lds(int n, int cols, int hs, int ntr) {
  const size_t ts = tt_stride(ntr);
  return sizeof(double) * cols * ((5 + ts) * (n + 2 * hs) + (5 + 2 * ts) * (n + 1));
}

// Lines per work-group of a tile, and its modelled cost per cell in waves of
// full lanes: the idle lanes of the waves, the waves a CU holds (16, by the
// registers; work-groups of 5 to 8 waves fit twice, larger ones and those that
// fill the LDS once, and a lone group idles at its barriers), and in y and z the
// runs of `cols` neighbouring lines that a load covers.  Measured, y at
// 256x256x128 with 3 tracers: 1 line 791 us, 2 (8 waves) 662, 3 (12 waves) 953, 4
// (16 waves) 856; z: 1 line 1110, 2 747, 3 (6 waves) 974, 4 (8 waves) 670, 5 (10
// waves) 1065, 6 (12 waves) 915, 8 (16 waves) 835.
struct TtCut {
  int cols;
  double cost;
};
inline TtCut tt_cut(int dir, int n, int64_t lines, int hs, int ntr) {
  TtCut best{0, 1e300};
  for (int m = 1; m * n <= TT_MAX && (m == 1 || (lines + m - 1) / m >= 256); m++) {
    const int waves = (m * n + 63) / 64;
    if (dir == 0 && pairs_collide(n, m, lines)) continue;
    const size_t lds = tt_lds(n, m, hs, ntr);
    if (lds > 160 * 1024) break;
    const int groups = (int)std::min<size_t>(waves <= 4 ? 16 / waves : waves <= 8 ? 2 : 1, 160 * 1024 / lds);
    const double runs = dir == 0 || m >= 4 ? 1.0 : m == 3 ? 1.05 : m == 2 ? 1.11 : 1.33;
    // a small grid needs fewer waves than a CU holds, but whole rounds of groups
    const double need = std::min(16.0, (double)lines * n / 64 / 256);
    const double held = std::max(1.0, need / (groups * waves)) * (groups == 1 ? 1.4 : 1.0);
    const int64_t wgs = (lines + m - 1) / m;
    const double rounds = wgs <= 1024 && wgs >= 256 ? (wgs + 255) / 256 * 256.0 / wgs : 1.0;
    const double cost = 64.0 * waves / (m * n) * held * rounds * runs * (waves == 1 ? 1.06 : waves == 2 ? 1.03 : 1.0);
    if (cost < best.cost * 0.999) best = TtCut{m, cost};
  }
  return best;
}

// Tile or walker for y and z lines, of `groups` walker work-groups: the walker's
// waves take steps of 64 cells of a line, the tile pays for idle lanes and short runs
// but not for the walker's head, tail and carries.  Around the line at (5, 3): y at n =
// 256 (cost 1.11 of the walker's) 662 against 704 us, 210 (1.33) 225 and 240, 150 (1.42)
// 486 and 552, 400 (1.5) 78 and 71, 300 (1.6) 607 and 422; z at 128 (1.0) 670 and 777,
// 150 (1.42) 577 and 566, 180 (1.42) 238 and 230.  The walker of (3, 2) gains more on its
// tile where that takes single y lines and there are few tracers (so that the walker's
// LDS lets a CU hold its waves), once the grid fills the chip: 39x456x215 with one tracer
// 303 (tile) and 231 us, 92x449x80 with three 364 and 287, 59x189x181 with three 171 and
// 157; but with five 520 and 594 at 237x147x116.  Two tracers take the tile's LDS of
// three and leave it behind by pairs of lines as well (cost 1.11): 156x228x160 398 and 368
// us, 288x237x52 250 and 221, where one and three are even or ahead (66x210x76 80 and
// 106).  A grid with fewer walker groups than CUs waits for one walk: 17x520x10 with five
// tracers 24 (tile) and 91 us, 57x6x388 with eight 48 and 101 (z).
inline bool tt_tile(const TtCut& cut, int dir, int ord, int n, int64_t groups, int ntr) {
  if (groups <= 192) return true;
  const double walker = (n + 63) / 64 * 64.0 / n;
  const bool quick = ord == 3 && ntr < 4 && groups > 1024;
  const double line = dir == 2 ? 1.3 : !quick ? 1.45 : ntr == 2 ? 1.05 : 1.3;
  return cut.cost < line * walker;
}

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
    if (pairs_collide(n, m, lines)) continue;
    const double e = slack[waves] * waves / m;
    if (e < cost) {
      cost = e;
      best = m;
    }
  }
  return best;
}

}  // namespace awfl_cut
