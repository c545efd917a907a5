// awfl_cell_pert.hpp -- the split-sweep numerics in FP32 perturbation form.
//
// The state is carried as FP32 deviations from the FP64 hydrostatic
// background: rho', rho*u, rho*v, rho*w, (rho theta)' -- the same variables
// the FP64 path stores.  WENO, the ADER differential transform and the
// Riemann flux run in FP32 on deviations wherever a full value would cancel:
//   * pressure only ever appears as p' = pbar ((1 + e)^GAMMA - 1),
//     e = (rho theta)'/(rho theta)bar, from a binomial series -- never as
//     C0 (rho theta)^GAMMA - pbar (catastrophic in FP32 at ~1e5 Pa);
//   * the x/y flux drops the level-constant background pressure (it cancels
//     exactly in the flux difference); the z flux is already written with the
//     background pressure subtracted (S:1628-1629, 2042);
//   * the characteristic decomposition and recomposition of the Riemann flux
//     are linear in the state for fixed eigen-parameters, so they are applied
//     to the deviation vector; the background recomposes to itself.
// Full density and rho*theta (background + deviation, FP32) appear only where
// the reference divides by them or forms products with them.  The FP64
// background enters as FP32 per-level / per-point constants.
#pragma once
#include <type_traits>

#include "awfl_cell.hpp"

namespace awfl {
namespace pert {

constexpr float C0F = (float)C0;
constexpr float GAMMAF = (float)GAMMA;
constexpr float GRAVF = (float)GRAV;

// (1 + e)^GAMMA - 1: binomial series (degree 5: the first omitted term is
// below 5e-9 of the result for |e| <= 1/16, a tenth of an FP32 ulp), else
// exp2/log2 of the hardware.
__device__ __forceinline__ float powm1_gamma(float e) {
  if (fabsf(e) <= 0.0625f) {
    float q = (float)BINOM_GAMMA.c[5];
    q = fmaf(q, e, (float)BINOM_GAMMA.c[4]);
    q = fmaf(q, e, (float)BINOM_GAMMA.c[3]);
    q = fmaf(q, e, (float)BINOM_GAMMA.c[2]);
    q = fmaf(q, e, (float)BINOM_GAMMA.c[1]);
    return q * e;
  }
  return __builtin_amdgcn_exp2f(GAMMAF * __builtin_amdgcn_logf(1.0f + e)) - 1.0f;
}

// background of one GLL point: density, rho*theta, pressure, 1/(rho theta)
struct PointBg {
  float r, rt, p, rrt;
};

template <int NGLL>
struct CellBgP {
  PointBg pt[NGLL];        // x/y: all points equal the level's cell averages (S:680, 697)
  bool wall_bot, wall_top; // z: solid wall and k == 0 / k == nz-1
};

// Launch constants in FP32.
struct SweepKF {
  float dt, rd;
  float ndt[KMAX];
  float tav[KMAX];
};

// n times the GLL derivative of point values (two or three points), and that
// added to the two edge values: gll_deriv / gll_deriv_edges of awfl_cell.hpp
template <int NGLL>
__device__ __forceinline__ void gll_deriv_f(const float (&F)[NGLL], float n, float (&d)[NGLL]) {
  static_assert(NGLL == 2 || NGLL == 3, "FP32 sweeps have two or three points");
  if constexpr (NGLL == 2) {
    d[0] = d[1] = (F[1] - F[0]) * n;
  } else {
    const float a = (F[2] - F[0]) * n, c = fmaf(-2.0f, F[1], F[0] + F[2]), h = 2.0f * n;
    d[0] = fmaf(-h, c, a);
    d[1] = a;
    d[2] = fmaf(h, c, a);
  }
}
template <int NGLL>
__device__ __forceinline__ void gll_deriv_edges_f(const float (&F)[NGLL], float n, float& eL, float& eR) {
  if constexpr (NGLL == 2) {
    const float t = (F[1] - F[0]) * n;
    eL += t;
    eR += t;
  } else {
    const float a = F[2] - F[0], c = fmaf(-2.0f, F[1], F[0] + F[2]), h = 2.0f * n;
    eL = fmaf(-h, c, fmaf(n, a, eL));
    eR = fmaf(h, c, fmaf(n, a, eR));
  }
}

// One cell of a DIR sweep in perturbation form: deviation stencils -> deviation
// edge states (time averaged) and the z gravity source.  The transform's
// organisation is cell_edges_of's (awfl_cell.hpp): the normal velocity's Taylor
// coefficients u_k carry every flux (u_k sums in place of the reference's
// quotients), the last level goes straight into the edge states, and the z
// source's cell average comes from the end points.
template <int ORD, int NGLL, int DIR>
__device__ __forceinline__ void cell_edges_pert(const float (&st)[5][ORD], const CellBgP<NGLL>& bg, bool weno_s,
                                                bool weno_w, const SweepKF& K, float (&eL)[5], float (&eR)[5],
                                                float& src_avg) {
  constexpr int NM = 1 + DIR;
  static_assert(NGLL <= 3, "one or two transform levels");
  float q[5][NGLL];              // level 0: deviations (full rho in r0, rho*theta in t0)
  float r0[NGLL], t0[NGLL], rr[NGLL], u0[NGLL], pp[NGLL];
  sfor<5>([&](auto l) { reconstruct<ORD, NGLL>(st[l], (l == idR || l == idT) ? weno_s : weno_w, q[l]); });
  const float sv = DIR == 2 ? -GRAVF * q[idR][NGLL - 1] : 0.0f;   // S:1439: the last point's, everywhere
  if constexpr (DIR == 2) {
    if (bg.wall_top) q[idW][NGLL - 1] = 0.0f;
    if (bg.wall_bot) q[idW][0] = 0.0f;
  }
  sfor<NGLL>([&](auto ii) {
    const PointBg& b = bg.pt[ii];
    r0[ii] = b.r + q[idR][ii];
    t0[ii] = b.rt + q[idT][ii];
    rr[ii] = __builtin_amdgcn_rcpf(r0[ii]);
    u0[ii] = q[NM][ii] * rr[ii];
    // p' at level 0; the constant-in-the-sweep background pressure has zero
    // derivative (x/y), z subtracts hyPressureGLL (S:2042): both leave p'
    pp[ii] = b.p * powm1_gamma(q[idT][ii] * b.rrt);
  });
  sfor<5>([&](auto l) {
    eL[l] = q[l][0];
    eR[l] = q[l][NGLL - 1];
  });
  float sa = sv;
  if constexpr (DIR == 2) sa = fmaf(-GRAVF * (K.tav[1] * K.ndt[0]), q[NM][NGLL - 1] - q[NM][0], sa);
  // level 1
  float d[5][NGLL];
  sfor<5>([&](auto l) {
    float F[NGLL];
    sfor<NGLL>([&](auto s) {
      if constexpr (l == idR) F[s] = q[NM][s];
      else if constexpr (l == NM) F[s] = fmaf(u0[s], q[NM][s], pp[s]);
      else F[s] = u0[s] * (l == idT ? t0[s] : q[l][s]);
    });
    if constexpr (NGLL == 2) {
      gll_deriv_edges_f<NGLL>(F, K.ndt[0] * K.tav[1], eL[l], eR[l]);
      if constexpr (DIR == 2 && l == idW) {
        eL[l] = fmaf(K.tav[1], sv, eL[l]);
        eR[l] = fmaf(K.tav[1], sv, eR[l]);
      }
    } else {
      gll_deriv_f<NGLL>(F, K.ndt[0], d[l]);
      if constexpr (DIR == 2 && l == idW) {       // S:2049-2055
        sfor<NGLL>([&](auto ii) { d[l][ii] += sv; });
        if (bg.wall_top) d[l][NGLL - 1] = 0.0f;
        if (bg.wall_bot) d[l][0] = 0.0f;
      }
      eL[l] = fmaf(d[l][0], K.tav[1], eL[l]);
      eR[l] = fmaf(d[l][NGLL - 1], K.tav[1], eR[l]);
    }
  });
  // level 2
  if constexpr (NGLL == 3) {
    float u1[NGLL], p1[NGLL];
    sfor<NGLL>([&](auto ii) {
      u1[ii] = fmaf(-d[idR][ii], u0[ii], d[NM][ii]) * rr[ii];
      p1[ii] = ((bg.pt[ii].p + pp[ii]) * __builtin_amdgcn_rcpf(t0[ii])) * (GAMMAF * d[idT][ii]);
    });
    if constexpr (DIR == 2) sa = fmaf(-GRAVF * (K.tav[2] * K.ndt[1]), d[NM][2] - d[NM][0], sa);
    sfor<5>([&](auto l) {
      float F[NGLL];
      sfor<NGLL>([&](auto s) {
        if constexpr (l == idR) F[s] = d[NM][s];
        else {
          F[s] = u0[s] * d[l][s];
          F[s] = fmaf(u1[s], l == idT ? t0[s] : q[l][s], F[s]);
          if constexpr (l == NM) F[s] += p1[s];
        }
      });
      gll_deriv_edges_f<NGLL>(F, K.ndt[1] * K.tav[2], eL[l], eR[l]);
      if constexpr (DIR == 2 && l == idW) {
        eL[l] = fmaf(-0.5f * GRAVF * K.tav[2], d[idR][0], eL[l]);
        eR[l] = fmaf(-0.5f * GRAVF * K.tav[2], d[idR][NGLL - 1], eR[l]);
      }
    });
  }
  if constexpr (DIR == 2) {
    if (bg.wall_top) eR[idW] = 0.0f;
    if (bg.wall_bot) eL[idW] = 0.0f;
  }
  src_avg = sa;
}

// background seen by one face
struct FaceBgP {
  float r, rt, p, rrt;     // density, rho*theta, pressure, 1/(rho theta) at the face
  float pq, rq, bq;        // y flux only: p and 1/B of B = r*rt (its average of conservatives)
};

// Upwind characteristic flux in perturbation form: deviation edge states
// -> flux whose difference gives the tendency (normal-momentum flux without
// the face background pressure).
template <int DIR>
__device__ __forceinline__ void riemann_pert(const float (&L)[5], const float (&R)[5], const FaceBgP& fb,
                                             float (&F)[5]) {
  constexpr int NM = 1 + DIR;
  constexpr int T1 = DIR == 0 ? 2 : 1;
  constexpr int T2 = DIR == 2 ? 2 : 3;
  float rL = fb.r + L[0], rR = fb.r + R[0];
  float tL = fb.rt + L[4], tR = fb.rt + R[4];
  float r = 0.5f * (rL + rR);
  float un, ut1, ut2, t, e;
  if constexpr (DIR == 1) {       // averages of conservative variables (S:1210-1214)
    un = 0.5f * (L[NM] + R[NM]);
    ut1 = 0.5f * (L[T1] + R[T1]);
    ut2 = 0.5f * (L[T2] + R[T2]);
    t = 0.5f * (tL + tR);
    e = fmaf(r, t, -fb.bq) * fb.rq;
  } else {
    float iL = __builtin_amdgcn_rcpf(rL), iR = __builtin_amdgcn_rcpf(rR);
    un = 0.5f * (L[NM] * iL + R[NM] * iR);
    ut1 = 0.5f * (L[T1] * iL + R[T1] * iR);
    ut2 = 0.5f * (L[T2] * iL + R[T2] * iR);
    t = 0.5f * (tL * iL + tR * iR);
    e = fmaf(r, t, -fb.rt) * fb.rrt;
  }
  float pb = DIR == 1 ? fb.pq : fb.p;
  float p = pb + pb * powm1_gamma(e);
  // sound speed and its reciprocal from one hardware reciprocal square root
  const float c2 = GAMMAF * p * __builtin_amdgcn_rcpf(r);
  const float rc = __builtin_amdgcn_rsqf(c2);
  const float cs = c2 * rc;
  const float i2c = 0.5f * rc;
  // the waves and the recomposed deviations in differences of the two sides
  // (riemann in awfl_cell.hpp): v the deviation that the acoustic waves and the
  // upwind side add to U
  const bool up = un > 0;
  const float u0 = up ? L[0] : R[0], u1 = up ? L[T1] : R[T1], u2 = up ? L[T2] : R[T2];
  const float D = fmaf(un, R[0] - L[0], L[NM] - R[NM]) * i2c;
  const float d = (R[4] - L[4]) * (0.5f * __builtin_amdgcn_rcpf(t));
  const float v = D + (up ? d : -d);
  const float q1 = u0 + v;                          // deviations of the recomposed state
  const float qn = fmaf(-cs, d, fmaf(un, q1 - 0.5f * (L[0] + R[0]), 0.5f * (L[NM] + R[NM])));
  const float q5 = fmaf(t, D, 0.5f * (L[4] + R[4]));
  const float un1 = qn * __builtin_amdgcn_rcpf(fb.r + q1);
  F[0] = qn;
  F[NM] = fmaf(qn, un1, fb.p * powm1_gamma(q5 * fb.rrt));
  F[T1] = un1 * fmaf(ut1, v, u1);
  F[T2] = un1 * fmaf(ut2, v, u2);
  F[4] = un1 * (fb.rt + q5);
}

}  // namespace pert
}  // namespace awfl
