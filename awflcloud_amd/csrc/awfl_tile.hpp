// awfl_tile.hpp -- the tile sweep: how one split sweep's cells, edge states and
// face fluxes pass between lanes, shared by the FP64 sweeps
// (awfl_dycore.hip) and the FP32 perturbation form (awfl_pert.hip).
//
// A work-group takes `cols` neighbouring lines along the sweep, whole or a
// segment of each, one lane per cell:
//   stage   the cells and hs cells beyond either end go to LDS, with the
//           periodic wrap or the wall rule applied at the load (S:631-662,
//           994-1025, 1351-1382; S = Spatial_euler3d_cons_expl_cart_fv_Agrid.h);
//   cells   a lane reconstructs and evolves its cell and puts the right edge
//           state into the slot of its high face;
//   faces   a lane takes the right edge state of the previous cell from the
//           slot of its low face, forms the flux and puts it back there (the
//           lane is the only reader and the only writer);
//   update  a lane takes its high face's flux from its slot and updates its
//           cell.
// A segment also reconstructs the neighbouring cell at either end, whose edge
// state its end faces need.  Every global read happens before the first
// barrier, so whole lines may be updated in place.
//
// What bounds it: instruction issue (and the clock the FP64 load leaves).  One
// cell per lane takes 96 registers in FP64 x and y, five waves per SIMD, and 112 in z,
// four.
// Work-groups are best four waves or fewer: the more of them a CU holds, the
// less a barrier costs (y at 256x256x128 in segments: 330 us with four waves,
// 371 with seven, 396 with six).  LDS holds a cell's 5 values contiguously:
// every stencil address is one base plus a constant, and lanes 5 elements
// apart meet no bank twice.  Walking a line in chunks of such a tile, with the
// chunk's last edge state and flux carried over, would save the segments'
// second reconstructions, but its loop takes the FP64 kernel to 144-168
// registers (spills at 128).
#pragma once
#include "awfl_cut.hpp"
#include "awfl_internal.hpp"
#include "awfl_tables.hpp"

namespace awfl_tile {

using awfl::sfor;

using awfl_cut::TilePlan;

// P supplies the scalar (P::real), ORD, DIR, TX (lines of a y or z tile, x
// fastest; x tiles take p.cols lines along y), and over its arguments A:
//   in() the state read, G() the grid,
//   cell(o, a, st, eL, eR, src)     stencils of cell a -> edge states, z source
//   face(o, line, f, qL, qR, F)     flux of face f
//   wall(o, line, f, q, F)          flux of a wall face with edge state q
//   put(o, line, a, at, cell, F0, F1, src)   update of cell a at state offset at
// (o: the level of x and y tiles, j of z tiles).
template <class P>
__device__ __forceinline__ void sweep(const P& A, const TilePlan& T) {
  using real = typename P::real;
  constexpr int DIR = P::DIR, TX = P::TX, hs = (P::ORD - 1) / 2;
  constexpr int NM = 1 + DIR;
  extern __shared__ double smem_[];
  real* const sm = reinterpret_cast<real*>(smem_);
  const auto& G = A.G();
  const real* const in = A.in();
  const int n = DIR == 0 ? G.nx : DIR == 1 ? G.ny : G.nz;
  const int cols = DIR == 0 ? T.cols : TX;
  const int rows = T.rows;
  const bool per = G.bc[DIR] == AWFL_BC_PERIODIC;
  const bool full = T.nseg == 1;
  const dim3 tb = tile_coords();
  const int o = tb.y;
  const int s0 = tb.z * T.seglen, s1 = min(n, s0 + T.seglen);
  const int lo = full || (!per && s0 == 0) ? s0 : s0 - 1;
  const int nrow = (full || (!per && s1 == n) ? s1 : s1 + 1) - lo;
  // lane -> column c, row r (cell a of the line)
  const int t = threadIdx.x;
  int c, r;
  if constexpr (DIR == 0) {
    c = cols == 1 ? 0 : t / rows;
    r = t - c * rows;
  } else {
    c = t % TX;
    r = t / TX;
  }
  const int nline = DIR == 0 ? G.ny : G.nx;
  const int line = tb.x * cols + c;
  const bool act = c < cols && line < nline && r < nrow;
  const int a = lo + r;
  const int64_t sa = DIR == 0 ? 1 : DIR == 1 ? G.sy : G.sz;
  auto line_base = [&](int l) -> int64_t {
    if constexpr (DIR == 0) return (int64_t)(hs + o) * G.sz + (int64_t)(hs + l) * G.sy + hs;
    else if constexpr (DIR == 1) return (int64_t)(hs + o) * G.sz + (int64_t)hs * G.sy + hs + l;
    else return (int64_t)hs * G.sz + (int64_t)(hs + o) * G.sy + hs + l;
  };
  // LDS: row p of column cc of the staged cells (p from -hs) and of the slots
  // (slot p: low face of row p)
  auto st_at = [&](int cc, int p) { return 5 * (DIR == 0 ? cc * (rows + 2 * hs) + p + hs : (p + hs) * TX + cc); };
  auto e_at = [&](int cc, int p) { return 5 * (DIR == 0 ? cc * (rows + 1) + p : p * TX + cc); };
  real* const s_st = sm;
  real* const s_e = s_st + 5 * cols * (rows + 2 * hs);

  // stage; source: stored cell of logical index v of the line (zn: a wall's
  // clamped cell, whose normal momentum is zero)
  auto source = [&](int v, bool& zn) {
    zn = false;
    if (v >= 0 && v < n) return v;
    if (per) {
      if (n > hs + 1) return v < 0 ? v + n : v - n;    // a tile reaches at most hs + 1 cells past the line
      const int w = v % n;
      return w < 0 ? w + n : w;
    }
    zn = true;
    return v < 0 ? 0 : n - 1;
  };
  real own[5];
  if (act) {                                           // (a row of a line is never clamped)
    bool zn;
    const int64_t g = line_base(line) + source(a, zn) * sa;
    sfor<5>([&](auto l) { own[l] = in[l * G.sl + g]; });
  }
  for (int h = t; h < 2 * hs * cols; h += blockDim.x) {
    int hc, hp;                                        // column, and which of the 2 hs cells beyond the rows
    if constexpr (DIR == 0) {
      hc = h / (2 * hs);
      hp = h % (2 * hs);
    } else {
      hc = h % TX;
      hp = h / TX;
    }
    if ((int)tb.x * cols + hc < nline) {
      const int p = hp < hs ? hp - hs : nrow + hp - hs;
      bool zn;
      const int64_t g = line_base(tb.x * cols + hc) + source(lo + p, zn) * sa;
      real v[5];
      sfor<5>([&](auto l) { v[l] = in[l * G.sl + g]; });
      if (zn) v[NM] = 0;
      sfor<5>([&](auto l) { s_st[st_at(hc, p) + l] = v[l]; });
    }
  }
  if (act) sfor<5>([&](auto l) { s_st[st_at(c, r) + l] = own[l]; });
  __syncthreads();

  // cells
  real eL[5], eR[5], src = 0;
  if (act) {
    real st[5][P::ORD];
    const real* w = s_st + st_at(c, r - hs);
    constexpr int step = DIR == 0 ? 5 : 5 * TX;
    sfor<5>([&](auto l) { sfor<P::ORD>([&](auto s) { st[l][s] = w[s * step + l]; }); });
    A.cell(o, a < 0 ? a + n : a >= n ? a - n : a, st, eL, eR, src);
    sfor<5>([&](auto l) { s_e[e_at(c, r + 1) + l] = eR[l]; });
  }
  __syncthreads();

  // faces.  A whole periodic line's first face has its last cell's edge state
  // on the left and, in x and y, is its face n too; the background of a
  // periodic z line's face n differs from face 0's (S:1628-1629), so that both
  // are formed.
  const bool ring = full && per;
  real F[5];
  if (act && a >= 0) {
    const bool wall_lo = !per && a == 0;
    const bool wrap = ring && r == 0;
    if (r > 0 || wrap || wall_lo) {
      const int slot = e_at(c, wrap ? nrow : r);
      real qL[5];
      sfor<5>([&](auto l) { qL[l] = wall_lo ? eL[l] : s_e[slot + l]; });
      A.face(o, line, a, qL, eL, F);
      if (DIR == 2 && wrap) {
        real Fn[5];
        A.face(o, line, n, qL, eL, Fn);
        sfor<5>([&](auto l) { s_e[slot + l] = Fn[l]; });
      } else if (!wall_lo) {
        sfor<5>([&](auto l) { s_e[slot + l] = F[l]; });
      }
    }
    if (!per && a == n - 1) {
      real Fn[5];
      A.wall(o, line, n, eR, Fn);
      sfor<5>([&](auto l) { s_e[e_at(c, r + 1) + l] = Fn[l]; });
    }
  }
  __syncthreads();

  // update
  if (act && a >= s0 && a < s1) {
    real F1[5], cell[5];
    sfor<5>([&](auto l) {
      F1[l] = s_e[e_at(c, r + 1) + l];
      cell[l] = s_st[st_at(c, r) + l];
    });
    A.put(o, line, a, line_base(line) + a * sa, cell, F, F1, src);
  }
}

}  // namespace awfl_tile
