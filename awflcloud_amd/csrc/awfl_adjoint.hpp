// awfl_adjoint.hpp -- tangent-linear and adjoint (reverse) forms of the
// per-cell and per-face numerics of one FP64 split sweep.
//
// The split sweep out = in + dt * T(in) of the forward kernels is a chain of
//   stencil (5 variables x ORD cells) -> WENO -> GLL values -> ADER
//   differential transform -> time-averaged edge states (and the z gravity
//   source), then per face the upwind characteristic flux, then the flux
//   difference.
// cell_fwd / riemann_fwd restate that chain for a generic scalar T; with
// T = Dual (value + one directional derivative) they give the exact
// tangent-linear map.  cell_adj / riemann_adj are the hand-written reverse
// sweeps (vector-Jacobian products), used by the adjoint kernels; they follow
// the production forward's statements (awfl_cell.hpp), which need fewer
// operations than the generic ones: WENO5 in differences, the transform by
// velocity Taylor coefficients, the flux in differences of the two sides.
// Against reverses of the generic statements the y line kernel went from
// 4,185 to about 2,400 FP64 operations per cell, and a gradient over 20 steps
// of 128x128x64 from 14.2 to 12.5 ms.  Everything here is host+device so that a host unit test
// can pin the reverse against the tangent (dot-product test) and the tangent
// against finite differences of the production forward (cell_edges/riemann).
#pragma once
#include "awfl_cell.hpp"

namespace awfl {
namespace adj {

#define AWFL_HD __host__ __device__ __forceinline__

// ---------------------------------------------------------------------------
// forward-mode scalar
// ---------------------------------------------------------------------------
struct Dual {
  double v, d;
  AWFL_HD constexpr Dual() : v(0.0), d(0.0) {}
  AWFL_HD constexpr Dual(double x) : v(x), d(0.0) {}
  AWFL_HD constexpr Dual(double x, double dx) : v(x), d(dx) {}
  AWFL_HD Dual& operator+=(const Dual& o) { v += o.v; d += o.d; return *this; }
  AWFL_HD Dual& operator-=(const Dual& o) { v -= o.v; d -= o.d; return *this; }
  AWFL_HD Dual& operator*=(const Dual& o) { d = d * o.v + v * o.d; v *= o.v; return *this; }
};
AWFL_HD constexpr Dual operator+(const Dual& a, const Dual& b) { return Dual(a.v + b.v, a.d + b.d); }
AWFL_HD constexpr Dual operator-(const Dual& a, const Dual& b) { return Dual(a.v - b.v, a.d - b.d); }
AWFL_HD constexpr Dual operator-(const Dual& a) { return Dual(-a.v, -a.d); }
AWFL_HD constexpr Dual operator*(const Dual& a, const Dual& b) { return Dual(a.v * b.v, a.d * b.v + a.v * b.d); }
AWFL_HD constexpr bool operator!=(const Dual& a, const Dual& b) { return a.v != b.v; }
AWFL_HD constexpr bool operator==(const Dual& a, const Dual& b) { return a.v == b.v; }
AWFL_HD constexpr bool operator>(const Dual& a, const Dual& b) { return a.v > b.v; }

AWFL_HD double val(double x) { return x; }
AWFL_HD double val(const Dual& x) { return x.v; }

AWFL_HD double rcp_g(double x) { return rcp(x); }
AWFL_HD Dual rcp_g(const Dual& x) {
  double r = rcp(x.v);
  return Dual(r, -x.d * r * r);
}
AWFL_HD double pow_g(double x) { return pow_gamma(x); }
AWFL_HD Dual pow_g(const Dual& x) {
  double p = pow_gamma(x.v);
  return Dual(p, GAMMA * p * rcp(x.v) * x.d);
}
// x^GAMMA near a background value B with known power (PowRef, as the
// production kernels): B^GAMMA (1 + (x-B)/B)^GAMMA
AWFL_HD double pow_at(double x, const PowRef& pr) { return pow_gamma_near(x, (x - pr.b) * pr.rb, pr.h, pr.l); }
AWFL_HD Dual pow_at(const Dual& x, const PowRef& pr) {
  double p = pow_gamma_near(x.v, (x.v - pr.b) * pr.rb, pr.h, pr.l);
  return Dual(p, GAMMA * p * rcp(x.v) * x.d);
}
AWFL_HD double sqrt_g(double x) { return sqrt(x); }
AWFL_HD Dual sqrt_g(const Dual& x) {
  double s = sqrt(x.v);
  return Dual(s, 0.5 * x.d * rcp(s));
}

// a b + c d with the value rounded as the production face averages round it
// (face_averages in awfl_cell.hpp), so that the upwind test sees the same sign
AWFL_HD double dot2(double a, double b, double c, double d) { return fma(a, b, c * d); }
AWFL_HD Dual dot2(const Dual& a, const Dual& b, const Dual& c, const Dual& d) {
  return Dual(fma(a.v, b.v, c.v * d.v), a.d * b.v + a.v * b.d + c.d * d.v + c.v * d.d);
}

// the WENO of weno_coefs for T = Dual takes its generic (non-double) branch,
// which calls rcp_t (found here by argument-dependent lookup)
AWFL_HD Dual rcp_t(const Dual& x) { return rcp_g(x); }

// ---------------------------------------------------------------------------
// differential-transform levels of one cell, kept for the reverse sweep
// ---------------------------------------------------------------------------
template <int NGLL, class T>
struct Tape {
  T q[5][NGLL][NGLL];      // [var][level][point]; level 0 full state (background added)
  T f[4][NGLL][NGLL];      // q_nm * var_l / r, l = 1..4
  T g[NGLL][NGLL];         // (r t)^gamma, levels >= 1 doubled
  T rr[NGLL], rrt[NGLL];   // 1/r, 1/(r t) at level 0
};

// WENO stage of one cell: the 5 reconstructions to the GLL points
// (deviations from the background)
template <int ORD, int NGLL, class T>
AWFL_HD void cell_recon(const T (&st)[5][ORD], bool weno_s, bool weno_w, T (&q0)[5][NGLL]) {
  sfor<5>([&](auto l) { reconstruct<ORD, NGLL>(st[l], (l == idR || l == idT) ? weno_s : weno_w, q0[l]); });
}

// Transform stage of one cell, generic scalar: from the reconstructed GLL
// values, the statements of cell_edges (awfl_cell.hpp) with pow/rcp/sqrt
// through pow_g/rcp_g.
template <int NGLL, int DIR, class T>
AWFL_HD void cell_dt(const T (&q0)[5][NGLL], const CellBg<NGLL>& bg, const SweepK& K, Tape<NGLL, T>& tp,
                     T (&eL)[5], T (&eR)[5], T& src_avg) {
  constexpr int NA = NGLL;
  constexpr int NM = 1 + DIR;
  auto& q = tp.q;
  auto& f = tp.f;
  auto& g = tp.g;
  T src[NA][NGLL];
  sfor<5>([&](auto l) { sfor<NGLL>([&](auto ii) { q[l][0][ii] = q0[l][ii]; }); });
  sfor<NGLL>([&](auto ii) {
    if constexpr (DIR == 2) {
      q[idR][0][ii] += T(bg.rG[ii]);
      q[idT][0][ii] += T(bg.rtG[ii]);
    } else {
      q[idR][0][ii] += T(bg.r);
      q[idT][0][ii] += T(bg.rt);
    }
  });
  if constexpr (DIR == 2) {
    if (bg.wall_top) q[idW][0][NGLL - 1] = T(0.0);
    if (bg.wall_bot) q[idW][0][0] = T(0.0);
  }
  T sv = T(0.0);
  sfor<NGLL>([&](auto ii) {
    // 1/rho and 1/(rho theta) from one reciprocal of their product
    const T z = rcp_g(q[idR][0][ii] * q[idT][0][ii]);
    tp.rr[ii] = q[idT][0][ii] * z;
    tp.rrt[ii] = q[idR][0][ii] * z;
    sfor<4>([&](auto m) { f[m][0][ii] = q[NM][0][ii] * q[m + 1][0][ii] * tp.rr[ii]; });
    g[0][ii] = pow_at(q[idT][0][ii], DIR == 2 ? bg.ptG[ii] : bg.pt);
    if constexpr (DIR == 2) sv = -(q[idR][0][ii] - T(bg.rG[ii])) * T(GRAV);
  });
  if constexpr (DIR == 2) {
    sfor<NA>([&](auto kt) { sfor<NGLL>([&](auto ii) { src[kt][ii] = sv; }); });
  }
  sfor<NA - 1>([&](auto kt) {
    constexpr double rkt1 = 1.0 / (kt + 1.0);
    const T ndt = T(K.ndt[kt]);
    sfor<NGLL>([&](auto ii) {
      T d[5];
      sfor<5>([&](auto l) { d[l] = T(0.0); });
      sfor<NGLL>([&](auto s) {
        constexpr double D = Deriv<NGLL>::m[s][ii];
        if constexpr (D == 0.0) return;
        d[0] += T(D) * q[NM][kt][s];
        sfor<4>([&](auto m) {
          constexpr int l = m + 1;
          if constexpr (l == NM) {
            if constexpr (kt == 0) {
              if constexpr (DIR == 2) d[l] += T(D) * (f[m][kt][s] + T(C0) * g[kt][s] - T(bg.pG[s]));
              else d[l] += T(D) * (f[m][kt][s] + T(C0) * g[kt][s]);
            } else {
              d[l] += T(D) * (f[m][kt][s] + T(0.5 * C0) * g[kt][s]);
            }
          } else {
            d[l] += T(D) * f[m][kt][s];
          }
        });
      });
      sfor<5>([&](auto l) {
        if constexpr (DIR == 2 && l == idW) q[l][kt + 1][ii] = d[l] * ndt + src[kt][ii] * T(rkt1);
        else q[l][kt + 1][ii] = d[l] * ndt;
      });
      if constexpr (DIR == 2) {
        if (bg.wall_top) q[idW][kt + 1][NGLL - 1] = T(0.0);
        if (bg.wall_bot) q[idW][kt + 1][0] = T(0.0);
        src[kt + 1][ii] = -q[idR][kt + 1][ii] * T(GRAV);
      }
    });
    if constexpr (kt + 2 < NA) {
      sfor<NGLL>([&](auto ii) {
        sfor<4>([&](auto m) {
          constexpr int l = m + 1;
          T tot = T(0.0);
          sfor<kt + 2>([&](auto ir) {
            if constexpr (ir == 0) tot += q[NM][ir][ii] * q[l][kt + 1 - ir][ii];
            else tot += q[NM][ir][ii] * q[l][kt + 1 - ir][ii] - q[idR][ir][ii] * f[m][kt + 1 - ir][ii];
          });
          f[m][kt + 1][ii] = tot * tp.rr[ii];
        });
        T tg = T(0.0);
        sfor<kt + 1>([&](auto ir) {
          constexpr double wgt = kt + 1.0 - ir;
          if constexpr (ir == 0)
            tg += T(wgt) * (T(GAMMA) * g[ir][ii] * q[idT][kt + 1 - ir][ii]);
          else
            tg += T(wgt) * (T(GAMMA) * g[ir][ii] * q[idT][kt + 1 - ir][ii] - q[idT][ir][ii] * g[kt + 1 - ir][ii]);
        });
        g[kt + 1][ii] = (T(GAMMA) * g[0][ii] * q[idT][kt + 1][ii] + tg * T(rkt1)) * tp.rrt[ii];
      });
    }
  });
  sfor<5>([&](auto l) {
    T a0 = q[l][0][0], a1 = q[l][0][NGLL - 1];
    sfor<NA - 1>([&](auto km) {
      constexpr int kt = km + 1;
      a0 += q[l][kt][0] * T(K.tav[kt]);
      a1 += q[l][kt][NGLL - 1] * T(K.tav[kt]);
    });
    eL[l] = a0;
    eR[l] = a1;
  });
  if constexpr (DIR == 2) {
    T sa = T(0.0);
    sfor<NGLL>([&](auto ii) {
      T s0 = src[0][ii];
      sfor<NA - 1>([&](auto km) {
        constexpr int kt = km + 1;
        s0 += src[kt][ii] * T(K.tav[kt]);
      });
      sa += s0 * T(Gll<NGLL>::wts[ii]);
    });
    src_avg = sa;
  } else {
    src_avg = T(0.0);
  }
}

// One cell of a DIR sweep, generic scalar: WENO stage then transform stage
template <int ORD, int NGLL, int DIR, class T>
AWFL_HD void cell_fwd(const T (&st)[5][ORD], const CellBg<NGLL>& bg, bool weno_s, bool weno_w, const SweepK& K,
                      Tape<NGLL, T>& tp, T (&eL)[5], T (&eR)[5], T& src_avg) {
  T q0[5][NGLL];
  cell_recon<ORD, NGLL>(st, weno_s, weno_w, q0);
  cell_dt<NGLL, DIR>(q0, bg, K, tp, eL, eR, src_avg);
}

// Upwind characteristic flux, generic scalar (statements of riemann in
// awfl_cell.hpp); p_face is the background pressure the z flux subtracts.
template <int DIR, class T>
AWFL_HD void riemann_fwd(const T (&L)[5], const T (&R)[5], const FaceRef& fr, double p_face, T (&F)[5]) {
  constexpr int NM = 1 + DIR;
  constexpr int T1 = DIR == 0 ? 2 : 1;
  constexpr int T2 = DIR == 2 ? 2 : 3;
  T r = T(0.5) * (L[0] + R[0]);
  T un, ut1, ut2, t, ir, hit;          // averages (face_averages), 1/r, 1/(2 t)
  if constexpr (DIR == 1) {
    un = T(0.5) * (L[NM] + R[NM]);
    ut1 = T(0.5) * (L[T1] + R[T1]);
    ut2 = T(0.5) * (L[T2] + R[T2]);
    t = T(0.5) * (L[4] + R[4]);
    const T z = rcp_g(r * t);
    ir = t * z;
    hit = (T(0.5) * r) * z;
  } else {
    const T LR = L[0] * R[0];
    const T x4 = dot2(L[4], R[0], R[4], L[0]);
    const T y = LR * x4, z = rcp_g(y * r), iy = z * r;
    ir = z * y;
    hit = LR * (iy * LR);
    const T h = T(0.5) * (iy * x4);
    un = dot2(L[NM], R[0], R[NM], L[0]) * h;
    ut1 = dot2(L[T1], R[0], R[T1], L[0]) * h;
    ut2 = dot2(L[T2], R[0], R[T2], L[0]) * h;
    t = x4 * h;
  }
  T cs = sqrt_g(T(GAMMA * C0) * pow_at(r * t, fr.rt) * ir);
  T i2c = T(0.5) * rcp_g(cs);
  const bool up = val(un) > 0;
  const T(&U)[5] = up ? L : R;
  T D = (un * (R[0] - L[0]) + (L[NM] - R[NM])) * i2c;
  T d = (R[4] - L[4]) * hit;
  T v = up ? D + d : D - d;
  T q1 = U[0] + v;
  T qn = (un * (q1 - r) + T(0.5) * (L[NM] + R[NM])) - cs * d;
  T q5 = T(0.5) * (L[4] + R[4]) + t * D;
  T un1 = qn * rcp_g(q1);
  F[0] = qn;
  F[NM] = qn * un1 + T(C0) * pow_at(q5, fr.q5);
  if constexpr (DIR == 2) F[NM] -= T(p_face);
  F[T1] = un1 * (U[T1] + ut1 * v);
  F[T2] = un1 * (U[T2] + ut2 * v);
  F[4] = un1 * q5;
}

// ---------------------------------------------------------------------------
// reverse sweeps (FP64)
// ---------------------------------------------------------------------------

// Lb += (dF/dL)^T Fb, Rb += (dF/dR)^T Fb at the state (L, R)
template <int DIR>
AWFL_HD void riemann_adj(const double (&L)[5], const double (&R)[5], const FaceRef& fr, const double (&Fb)[5],
                         double (&Lb)[5], double (&Rb)[5]) {
  constexpr int NM = 1 + DIR;
  constexpr int T1 = DIR == 0 ? 2 : 1;
  constexpr int T2 = DIR == 2 ? 2 : 3;
  // primal
  const FaceAvg av = face_averages<DIR>(L, R);
  const double r = av.r, un = av.un, ut1 = av.ut1, ut2 = av.ut2, t = av.t, hit = av.hit;
  const double it = 2.0 * hit;
  const double cs2 = (GAMMA * C0) * pow_at(r * t, fr.rt) * av.ir;
  double cs, i2c;
  sqrt_halfrsqrt(cs2, cs, i2c);        // as the forward riemann
  const bool up = un > 0;
  const double dR0 = R[0] - L[0];
  const double D = fma(un, dR0, L[NM] - R[NM]) * i2c;
  const double d = (R[4] - L[4]) * hit;
  const double v = D + (up ? d : -d);
  const double q1 = (up ? L[0] : R[0]) + v;
  const double qn = fma(-cs, d, fma(un, q1 - r, 0.5 * (L[NM] + R[NM])));
  const double q5 = fma(t, D, 0.5 * (L[4] + R[4]));
  const double z15 = rcp(q1 * q5);     // 1/q1 and 1/q5 from one reciprocal
  const double iq1 = q5 * z15;
  const double un1 = qn * iq1;
  const double y1 = (up ? L[T1] : R[T1]) + ut1 * v, y2 = (up ? L[T2] : R[T2]) + ut2 * v;
  // reverse, in the order of the statements backward
  const double un1b = Fb[NM] * qn + Fb[T1] * y1 + Fb[T2] * y2 + Fb[4] * q5;
  const double qnb = Fb[0] + Fb[NM] * un1 + un1b * iq1;
  const double y1b = Fb[T1] * un1, y2b = Fb[T2] * un1;
  const double q5b = Fb[4] * un1 + Fb[NM] * ((GAMMA * C0) * pow_at(q5, fr.q5)) * (q1 * z15);
  double q1b = qnb * un - un1b * (un1 * iq1);
  const double vb = y1b * ut1 + y2b * ut2 + q1b;
  const double Db = q5b * t + vb;
  const double db = (up ? vb : -vb) - qnb * cs;
  const double yD = Db * i2c, x4 = db * hit, h5 = 0.5 * q5b, hn = 0.5 * qnb;
  const double unb = qnb * (q1 - r) + yD * dR0;
  // cs through q_n and D (1/(2 cs)); cs^2 = C0 GAMMA (r t)^GAMMA / r
  const double c2b = (-qnb * d - (Db * D) * (2.0 * i2c)) * i2c * cs2;
  const double hrb = 0.5 * ((GAMMA - 1.0) * av.ir * c2b - qnb * un);   // half of r's adjoint
  const double tb = q5b * D - (db * d) * it + (GAMMA * it) * c2b;
  const double ut1b = y1b * v, ut2b = y2b * v, yu = yD * un;
  // upwind side
  Lb[0] += up ? q1b : 0.0;
  Rb[0] += up ? 0.0 : q1b;
  Lb[T1] += up ? y1b : 0.0;
  Rb[T1] += up ? 0.0 : y1b;
  Lb[T2] += up ? y2b : 0.0;
  Rb[T2] += up ? 0.0 : y2b;
  // averages
  if constexpr (DIR == 1) {
    const double hu = 0.5 * unb, ht = 0.5 * tb;
    Lb[0] += hrb - yu;
    Rb[0] += hrb + yu;
    Lb[NM] += (hn + yD) + hu;
    Rb[NM] += (hn - yD) + hu;
    Lb[T1] += 0.5 * ut1b;
    Rb[T1] += 0.5 * ut1b;
    Lb[T2] += 0.5 * ut2b;
    Rb[T2] += 0.5 * ut2b;
    Lb[4] += (h5 - x4) + ht;
    Rb[4] += (h5 + x4) + ht;
  } else {
    const double iL = R[0] * av.iLR, iR = L[0] * av.iLR;   // 1/L_0, 1/R_0
    const double hL = 0.5 * iL, hR = 0.5 * iR;
    Lb[NM] += (hn + yD) + hL * unb;
    Rb[NM] += (hn - yD) + hR * unb;
    Lb[T1] += hL * ut1b;
    Rb[T1] += hR * ut1b;
    Lb[T2] += hL * ut2b;
    Rb[T2] += hR * ut2b;
    Lb[4] += (h5 - x4) + hL * tb;
    Rb[4] += (h5 + x4) + hR * tb;
    Lb[0] += (hrb - yu) - hL * iL * (unb * L[NM] + ut1b * L[T1] + ut2b * L[T2] + tb * L[4]);
    Rb[0] += (hrb + yu) - hR * iR * (unb * R[NM] + ut1b * R[T1] + ut2b * R[T2] + tb * R[4]);
  }
}

// Lb += (dF(L, L) / dL)^T Fb at a wall, whose face takes both sides from the
// boundary cell's edge state L (S:822-823, 1577-1578).  A consistent flux of
// two equal states is the physical flux of L (wall_flux), whose derivative
// riemann_adj forms term by term; here it takes a few operations.
template <int DIR>
AWFL_HD void wall_adj(const double (&L)[5], const FaceRef& fr, const double (&Fb)[5], double (&Lb)[5]) {
  constexpr int NM = 1 + DIR;
  constexpr int T1 = DIR == 0 ? 2 : 1;
  constexpr int T2 = DIR == 2 ? 2 : 3;
  const double z = rcp(L[0] * L[4]), iL = z * L[4];
  const double un = L[NM] * iL;
  const double p5 = C0 * pow_at(L[4], fr.q5);
  const double xb = fma(Fb[NM], L[NM], fma(Fb[T1], L[T1], fma(Fb[T2], L[T2], Fb[4] * L[4])));   // un's adjoint
  Lb[0] -= xb * un * iL;
  Lb[NM] += Fb[0] + fma(Fb[NM], un, xb * iL);
  Lb[T1] += Fb[T1] * un;
  Lb[T2] += Fb[T2] * un;
  Lb[4] += fma(Fb[4], un, Fb[NM] * GAMMA * p5 * (z * L[0]));
}

// tvb * d tv_eval<N>(a) / da, accumulated into ab
template <int N, int M>
AWFL_HD void tv_adj(const double (&a)[M], double tvb, double (&ab)[M]) {
  sfor<Tv<N>::n>([&](auto t) {
    constexpr int j = Tv<N>::j[t];
    constexpr int k = Tv<N>::k[t];
    constexpr double c = Tv<N>::c[t];
    if constexpr (j == k) {
      ab[j] += 2.0 * c * a[j] * tvb;
    } else {
      ab[j] += c * a[k] * tvb;
      ab[k] += c * a[j] * tvb;
    }
  });
}

// ub += (d reconstruct_w5 / du)^T gb, the reverse of the difference form
// (awfl_cell.hpp) with its names.  The weights' derivatives need 1/D_i and 1/e_i
// besides the normalisations: each group of four and its sum share one
// reciprocal.  228 operations against 344 of the general reverse.
AWFL_HD void reconstruct_w5_adj(const double (&u)[5], const double (&gb)[3], double (&ub)[5]) {
  const double d0 = u[1] - u[0], d1 = u[2] - u[1], d2 = u[3] - u[2], d3 = u[4] - u[3];
  const double s[3] = {d1 - d0, d2 - d1, d3 - d2};
  const double A[3] = {fma(2.0, d1, s[0]), d1 + d2, fma(2.0, d2, -s[2])};
  const double M = s[2] - s[0], Q = fma(-2.0, s[1], s[0] + s[2]);
  double t[4];
  sfor<3>([&](auto i) { t[i] = fma(kW5.tvs * s[i], s[i], A[i] * A[i]); });
  t[3] = fma(kW5.k1, t[1], kW5.k0 * (t[0] + t[2]));
  t[3] = fma(M, fma(kW5.m1, A[1], kW5.mm * M), t[3]);
  t[3] = fma(Q, fma(kW5.q1, s[1], kW5.qq * Q), t[3]);
  // first weights w_i = N_i / T, and 1/D_i = x_i / P
  double w[4], rD[4];
  {
    double D[4];
    sfor<4>([&](auto i) { D[i] = fma(t[i], t[i], kW5.eps); });
    const double D01 = D[0] * D[1], D23 = D[2] * D[3], P = D01 * D23;
    const double x[4] = {D[1] * D23, D[0] * D23, D01 * D[3], D01 * D[2]};
    const double N1 = kW5.c1 * x[1], N3 = kW5.c3 * x[3];
    const double T = fma(kW5.epsn, P, (x[0] + N1) + (x[2] + N3));
    const double z = rcp(P * T), rP = T * z, rT = P * z;
    sfor<4>([&](auto i) { rD[i] = x[i] * rP; });
    w[0] = x[0] * rT;
    w[1] = N1 * rT;
    w[2] = x[2] * rT;
    w[3] = N3 * rT;
  }
  // mapped weights W_i = G_i / S, and dm_i/dw_i over the sum
  double Wt[4], sl[4];
  {
    double a[4], e[4], x[4], G[4];
    weno_map<0, 5>(w[0], a[0], e[0]);
    weno_map<1, 5>(w[1], a[1], e[1]);
    weno_map<2, 5>(w[2], a[2], e[2]);
    weno_map<3, 5>(w[3], a[3], e[3]);
    const double e01 = e[0] * e[1], e23 = e[2] * e[3], P = e01 * e23;
    x[0] = e[1] * e23;
    x[1] = e[0] * e23;
    x[2] = e01 * e[3];
    x[3] = e01 * e[2];
    sfor<4>([&](auto i) { G[i] = a[i] * x[i]; });
    const double S = (G[0] + G[2]) + (G[1] + G[3]);
    const double z = rcp(P * S), rP = S * z, rS = P * z;
    sfor<4>([&](auto i) {
      constexpr double d = Weno<5>::idl[i];
      Wt[i] = G[i] * rS;
      // num' - m (1 - 2 d), m = G / P
      const double n1 = fma(w[i], fma(3.0, w[i], -6.0 * d), d + d * d);
      sl[i] = fma(-(1.0 - 2.0 * d) * rP, G[i], n1) * (x[i] * rS);
    });
  }
  // reverse: GLL values, weighted sums
  const double endb = gb[0] + gb[2], odb = 0.25 * (gb[2] - gb[0]);
  const double evb = fma(1.0 / 12.0, endb, (-1.0 / 24.0) * gb[1]);
  const double wQb = fma(kW5.ev_q, endb, kW5.md_q * gb[1]), wMb = kW5.od_m * odb;
  ub[2] += endb + gb[1];
  double Wb[4];
  sfor<3>([&](auto i) { Wb[i] = fma(odb, A[i], evb * s[i]); });
  Wb[3] = fma(wQb, Q, fma(wMb, M, Wb[1]));
  const double dot = fma(Wt[3], Wb[3], fma(Wt[2], Wb[2], fma(Wt[1], Wb[1], Wt[0] * Wb[0])));
  double wb[4];
  sfor<4>([&](auto i) { wb[i] = (Wb[i] - dot) * sl[i]; });
  const double dot1 = fma(w[3], wb[3], fma(w[2], wb[2], fma(w[1], wb[1], w[0] * wb[0])));
  // half the total variations' adjoints, negated: t_i w_i / D_i (wb_i - dot1)
  double h[4];
  sfor<4>([&](auto i) { h[i] = (t[i] * rD[i]) * (w[i] * (dot1 - wb[i])); });
  const double thb = 2.0 * h[3];
  double tb2[3];                       // twice the adjoints of t_0 .. t_2
  tb2[0] = fma(2.0 * kW5.k0, thb, 4.0 * h[0]);
  tb2[1] = fma(2.0 * kW5.k1, thb, 4.0 * h[1]);
  tb2[2] = fma(2.0 * kW5.k0, thb, 4.0 * h[2]);
  const double W13 = Wt[1] + Wt[3];
  const double Mb = fma(thb, fma(kW5.m1, A[1], (2.0 * kW5.mm) * M), wMb * Wt[3]);
  const double Qb = fma(thb, fma(kW5.q1, s[1], (2.0 * kW5.qq) * Q), wQb * Wt[3]);
  const double A0b = fma(tb2[0], A[0], odb * Wt[0]);
  const double A1b = fma(kW5.m1 * thb, M, fma(tb2[1], A[1], odb * W13));
  const double A2b = fma(tb2[2], A[2], odb * Wt[2]);
  const double s0b = fma(kW5.tvs * tb2[0], s[0], evb * Wt[0]) + ((Qb - Mb) + A0b);
  const double s1b = fma(kW5.q1 * thb, Q, fma(kW5.tvs * tb2[1], s[1], fma(-2.0, Qb, evb * W13)));
  const double s2b = fma(kW5.tvs * tb2[2], s[2], evb * Wt[2]) + ((Qb + Mb) - A2b);
  const double d1b = fma(2.0, A0b, A1b) + (s0b - s1b), d2b = fma(2.0, A2b, A1b) + (s1b - s2b);
  ub[0] += s0b;
  ub[1] -= s0b + d1b;
  ub[2] += d1b - d2b;
  ub[3] += d2b - s2b;
  ub[4] += s2b;
}

// ub += (d reconstruct / du)^T gb: WENO (weno_coefs, then the projection to
// GLL points) or the plain projection of the stencil
template <int ORD, int NGLL>
AWFL_HD void reconstruct_adj(const double (&u)[ORD], bool doweno, const double (&gb)[NGLL], double (&ub)[ORD]) {
  using P = Proj<ORD, NGLL>;
  if (!doweno) {
    sfor<NGLL>([&](auto ii) {
      sfor<ORD>([&](auto s) {
        constexpr double cf = P::s2g[s][ii];
        if constexpr (cf != 0) ub[s] += cf * gb[ii];
      });
    });
    return;
  }
  if constexpr (ORD == 5 && NGLL == 3 && !(AWFL_PARITY & AWFL_PAR_BRIDGE)) {
    reconstruct_w5_adj(u, gb, ub);
    return;
  }
  using W = Weno<ORD>;
  constexpr int hs = W::hs;
  constexpr int NP = hs + 2;
  // primal: candidates, bridge, total variations, weights.  As in the
  // forward (reconstruct), the constant coefficients are never formed: the
  // GLL values are u_hs + sum_{c >= 1} kAvgProj[c][.] aw[c].
  double a[NP][ORD];
  sfor<hs + 1>([&](auto i) {
    a[i][0] = 0.0;
    sfor<hs + 1>([&](auto ii) {
      if constexpr (ii == 0) return;
      double t = 0.0;
      sfor<hs + 1>([&](auto s) {
        constexpr double cf = W::recon[i][s][ii];
        if constexpr (cf != 0) t += cf * u[i + s];
      });
      a[i][ii] = t;
    });
    sfor<ORD - hs - 1>([&](auto m) { a[i][hs + 1 + m] = 0.0; });
  });
  a[hs + 1][0] = 0.0;
  sfor<ORD>([&](auto ii) {
    if constexpr (ii == 0) return;
    double t = 0.0;
    sfor<ORD>([&](auto s) {
      constexpr double cf = kBridge<ORD>.m[s][ii];
      if constexpr (cf != 0) t += cf * u[s];
    });
    a[hs + 1][ii] = t;
  });
  double tv[NP];
  sfor<hs + 1>([&](auto i) {
    double ai[hs + 1];
    sfor<hs + 1>([&](auto ii) { ai[ii] = a[i][ii]; });
    tv[i] = tv_eval<hs + 1>(ai);
  });
  double tvhi = tv_eval<ORD>(a[hs + 1]);
  double lo = 0.0;
  sfor<hs + 1>([&](auto i) { lo += tv[i]; });
  lo *= 1.0 / (hs + 1);
  tv[hs + 1] = lo + (tvhi - lo) * W::sigma;
  // the NP reciprocals 1/(tv^2 + eps) and 1/(d^2 + w1 (1 - 2d)) each from
  // one reciprocal of the product and the products of the others
  double rDn[NP], b[NP], w1[NP], m[NP], w[NP], rden[NP];
  double R1, R2;
  {
    double D[NP], ex[NP], P;
    sfor<NP>([&](auto i) { D[i] = tv[i] * tv[i] + WENO_EPS; });
    excl_products<NP>(D, ex, P);
    // 1/P and 1/S1 = P / (eps P + sum_i d_i ex_i) from one reciprocal
    double N = 0.0;
    sfor<NP>([&](auto i) { N += W::idl[i] * ex[i]; });
    const double T1 = fma(WENO_EPS, P, N);
    const double z = rcp(P * T1);
    const double rP = T1 * z;
    R1 = P * P * z;
    sfor<NP>([&](auto i) {
      constexpr double d = W::idl[i];
      rDn[i] = ex[i] * rP;
      b[i] = d * rDn[i];
    });
  }
  {
    double E[NP], ex[NP], P;
    sfor<NP>([&](auto i) {
      constexpr double d = W::idl[i];
      w1[i] = b[i] * R1;
      E[i] = d * d + w1[i] * (1.0 - 2.0 * d);
    });
    excl_products<NP>(E, ex, P);
    // 1/P and 1/S2 from one reciprocal, as above
    double A[NP], M = 0.0;
    sfor<NP>([&](auto i) {
      constexpr double d = W::idl[i];
      A[i] = w1[i] * (d + d * d - 3.0 * d * w1[i] + w1[i] * w1[i]);
      M += A[i] * ex[i];
    });
    const double T2 = fma(WENO_EPS, P, M);
    const double z = rcp(P * T2);
    const double rP = T2 * z;
    R2 = P * P * z;
    sfor<NP>([&](auto i) {
      rden[i] = ex[i] * rP;
      m[i] = A[i] * rden[i];
    });
  }
  sfor<NP>([&](auto i) { w[i] = m[i] * R2; });
  // reverse: GLL projection (the centre cell's average takes the sum of the
  // GLL adjoints), weighted sum
  double awb[ORD];
  awb[0] = 0.0;
  sfor<NGLL>([&](auto ii) { ub[hs] += gb[ii]; });
  sfor<ORD>([&](auto s) {
    if constexpr (s == 0) return;
    double t = 0.0;
    sfor<NGLL>([&](auto ii) {
      constexpr double cf = kAvgProj<ORD, NGLL>.m[s][ii];
      if constexpr (cf != 0) t += cf * gb[ii];
    });
    awb[s] = t;
  });
  double ab[NP][ORD], wb[NP];
  sfor<NP>([&](auto i) {
    double t = 0.0;
    ab[i][0] = 0.0;
    sfor<ORD>([&](auto ii) {
      if constexpr (ii == 0) {
      } else if constexpr (i == hs + 1 || ii <= hs) {
        t += awb[ii] * a[i][ii];
        ab[i][ii] = w[i] * awb[ii];
      } else {
        ab[i][ii] = 0.0;
      }
    });
    wb[i] = t;
  });
  // second normalisation w = m / (sum m + eps)
  double dot = 0.0;
  sfor<NP>([&](auto i) { dot += wb[i] * w[i]; });
  double w1b[NP];
  sfor<NP>([&](auto i) {
    constexpr double d = W::idl[i];
    double mb = R2 * (wb[i] - dot);
    double x = w1[i];
    // m = num / den: m' = (num' - m (1 - 2d)) / den
    double dnum = d + d * d - 6.0 * d * x + 3.0 * x * x;
    w1b[i] = mb * (dnum - m[i] * (1.0 - 2.0 * d)) * rden[i];
  });
  // first normalisation w1 = b / (sum b + eps), b = idl / (tv^2 + eps)
  double dot1 = 0.0;
  sfor<NP>([&](auto i) { dot1 += w1b[i] * w1[i]; });
  double tvb[NP];
  sfor<NP>([&](auto i) {
    double bb = R1 * (w1b[i] - dot1);
    tvb[i] = -2.0 * bb * b[i] * tv[i] * rDn[i];
  });
  // sigma blend of the high-order indicator
  double tvhib = tvb[hs + 1] * W::sigma;
  double lob = tvb[hs + 1] * (1.0 - W::sigma) * (1.0 / (hs + 1));
  sfor<hs + 1>([&](auto i) {
    double ai[hs + 1], aib[hs + 1];
    sfor<hs + 1>([&](auto ii) {
      ai[ii] = a[i][ii];
      aib[ii] = 0.0;
    });
    tv_adj<hs + 1>(ai, tvb[i] + lob, aib);
    sfor<hs + 1>([&](auto ii) { ab[i][ii] += aib[ii]; });
  });
  tv_adj<ORD>(a[hs + 1], tvhib, ab[hs + 1]);
  // candidate and bridge polynomials (their constant coefficients, never
  // formed, pass nothing back)
  sfor<hs + 1>([&](auto i) {
    sfor<hs + 1>([&](auto ii) {
      if constexpr (ii == 0) return;
      sfor<hs + 1>([&](auto s) {
        constexpr double cf = W::recon[i][s][ii];
        if constexpr (cf != 0) ub[i + s] += cf * ab[i][ii];
      });
    });
  });
  sfor<ORD>([&](auto ii) {
    if constexpr (ii == 0) return;
    sfor<ORD>([&](auto s) {
      constexpr double cf = kBridge<ORD>.m[s][ii];
      if constexpr (cf != 0) ub[s] += cf * ab[hs + 1][ii];
    });
  });
}

// Fb[s] = sum_ii Deriv[s][ii] d[ii]: the derivative's transpose
template <int NGLL>
AWFL_HD void gll_deriv_t(const double (&d)[NGLL], double (&Fb)[NGLL]) {
  if constexpr (NGLL == 3) {           // rows -3 4 -1, -1 0 1, 1 -4 3
    const double e = d[0] - d[2];
    Fb[0] = fma(-2.0, d[0], -(e + d[1]));
    Fb[1] = 4.0 * e;
    Fb[2] = fma(2.0, d[2], d[1] - e);
  } else {
    sfor<NGLL>([&](auto s) {
      double t = 0.0;
      sfor<NGLL>([&](auto ii) {
        constexpr double D = Deriv<NGLL>::m[s][ii];
        if constexpr (D != 0.0) t += D * d[ii];
      });
      Fb[s] = t;
    });
  }
}

// q0b = (d (eL, eR, src_avg) / d q0)^T (eLb, eRb, srcb): reverse of the
// transform stage with the statements and names of cell_transform
// (awfl_cell.hpp), whose levels it recomputes from the GLL values q0.  The last
// level is linear in the fluxes of the level before and is never formed, and
// 1/r and 1/(r t) pass their adjoints on where they are used.  The two
// transverse momenta are carried by the velocity and act on nothing else, so
// each is transformed and reversed by itself, ahead of the others: its levels
// and those of the other variables' adjoints are never held together.
template <int NGLL, int DIR>
AWFL_HD void cell_dt_adj(const double (&q0)[5][NGLL], const CellBg<NGLL>& bg, const SweepK& K,
                         const double (&eLb)[5], const double (&eRb)[5], double srcb, double (&q0b)[5][NGLL]) {
  constexpr int NA = NGLL;
  constexpr int NM = 1 + DIR;
  constexpr int NL = NA - 1;           // levels formed
  constexpr int E = NGLL - 1;          // the high edge
  constexpr int T1 = DIR == 0 ? 2 : 1;
  constexpr int T2 = DIR == 2 ? 2 : 3;
  double q[5][NL][NGLL], u[NL][NGLL], g[NL][NGLL], rr[NGLL], rrt[NGLL];
  // levels 0 .. NA-2
  sfor<5>([&](auto l) { sfor<NGLL>([&](auto ii) { q[l][0][ii] = q0[l][ii]; }); });
  const double sv = DIR == 2 ? -GRAV * q[idR][0][E] : 0.0;
  sfor<NGLL>([&](auto ii) {
    const PowRef& pr = DIR == 2 ? bg.ptG[ii] : bg.pt;
    const double e = q[idT][0][ii] * pr.rb;
    q[idR][0][ii] += DIR == 2 ? bg.rG[ii] : bg.r;
    q[idT][0][ii] += DIR == 2 ? bg.rtG[ii] : bg.rt;
    g[0][ii] = pow_gamma_near(q[idT][0][ii], e, pr.h, pr.l);
  });
  if constexpr (DIR == 2) {
    if (bg.wall_top) q[idW][0][E] = 0.0;
    if (bg.wall_bot) q[idW][0][0] = 0.0;
  }
  sfor<NGLL>([&](auto ii) {
    const double r = q[idR][0][ii], rt = q[idT][0][ii], z = rcp(r * rt);
    rr[ii] = rt * z;
    rrt[ii] = r * z;
    u[0][ii] = q[NM][0][ii] * rr[ii];
  });
  // q[l][kt + 1] from the levels up to kt
  auto next_level = [&](auto l, auto kt) {
    constexpr double rkt1 = 1.0 / (kt + 1.0);
    double F[NGLL], d[NGLL];
    sfor<NGLL>([&](auto s) {
      if constexpr (l == idR) {
        F[s] = q[NM][kt][s];
      } else {
        double t = 0.0;
        if constexpr (l == NM) {
          if constexpr (kt == 0) t = DIR == 2 ? fma(C0, g[kt][s], -bg.pG[s]) : C0 * g[kt][s];
          else t = (0.5 * C0) * g[kt][s];
          t = fma(u[0][s], q[l][kt][s], t);
        } else {
          t = u[0][s] * q[l][kt][s];
        }
        sfor<kt>([&](auto j) { t = fma(u[j + 1][s], q[l][kt - 1 - j][s], t); });
        F[s] = t;
      }
    });
    gll_deriv<NGLL>(F, K.ndt[kt], d);
    sfor<NGLL>([&](auto ii) {
      if constexpr (DIR == 2 && l == idW) d[ii] = kt == 0 ? d[ii] + sv : fma(-GRAV * rkt1, q[idR][kt][ii], d[ii]);
      q[l][kt + 1][ii] = d[ii];
    });
  };
  sfor<NL - 1>([&](auto kt) {
    constexpr double rkt1 = 1.0 / (kt + 1.0);
    next_level(std::integral_constant<int, idR>{}, kt);
    next_level(std::integral_constant<int, NM>{}, kt);
    next_level(std::integral_constant<int, idT>{}, kt);
    if constexpr (DIR == 2) {
      if (bg.wall_top) q[idW][kt + 1][E] = 0.0;
      if (bg.wall_bot) q[idW][kt + 1][0] = 0.0;
    }
    sfor<NGLL>([&](auto ii) {
      double t = q[NM][kt + 1][ii];
      sfor<kt + 1>([&](auto j) { t = fma(-q[idR][j + 1][ii], u[kt - j][ii], t); });
      u[kt + 1][ii] = t * rr[ii];
      double tg = 0.0;
      sfor<kt + 1>([&](auto ir) {
        constexpr double wgt = kt + 1.0 - ir;
        double p = (GAMMA * g[ir][ii]) * q[idT][kt + 1 - ir][ii];
        if constexpr (ir > 0) p = fma(-q[idT][ir][ii], g[kt + 1 - ir][ii], p);
        tg = fma(wgt, p, tg);
      });
      g[kt + 1][ii] = fma(GAMMA * g[0][ii], q[idT][kt + 1][ii], tg * rkt1) * rrt[ii];
    });
  });
  // adjoints of the levels, from the time averages of the edge values (at a
  // wall every level of the normal momentum is zero there)
  double qb[5][NL][NGLL], ub[NL][NGLL], gb[NL][NGLL];
  double lb[5], hb[5], svb = 0.0;      // low- and high-edge adjoints
  auto averages = [&](auto l) {
    lb[l] = eLb[l];
    hb[l] = eRb[l];
    if constexpr (DIR == 2 && l == idW) {
      if (bg.wall_bot) lb[l] = 0.0;
      if (bg.wall_top) hb[l] = 0.0;
    }
    sfor<NL>([&](auto k) {
      const double w = k == 0 ? 1.0 : K.tav[k];
      sfor<NGLL>([&](auto ii) { qb[l][k][ii] = 0.0; });
      qb[l][k][0] = w * lb[l];
      qb[l][k][E] = w * hb[l];
    });
  };
  // the reverse of the fluxes at level kt behind q[l][kt + 1]
  auto flux_rev = [&](auto l, auto kt) {
    constexpr bool last = kt + 2 == NA;
    double d[NGLL], Fb[NGLL];
    if constexpr (last) {
      const double w = K.ndt[kt] * K.tav[kt + 1];
      sfor<NGLL>([&](auto ii) { d[ii] = 0.0; });
      d[0] = w * lb[l];
      d[E] = w * hb[l];
    } else {
      sfor<NGLL>([&](auto ii) { d[ii] = K.ndt[kt] * qb[l][kt + 1][ii]; });
    }
    gll_deriv_t<NGLL>(d, Fb);
    sfor<NGLL>([&](auto s) {
      if constexpr (l == idR) {
        qb[NM][kt][s] += Fb[s];
      } else {
        sfor<kt + 1>([&](auto j) {
          ub[j][s] = fma(Fb[s], q[l][kt - j][s], ub[j][s]);
          qb[l][kt - j][s] = fma(Fb[s], u[j][s], qb[l][kt - j][s]);
        });
        if constexpr (l == NM) gb[kt][s] = fma(Fb[s], kt == 0 ? C0 : 0.5 * C0, gb[kt][s]);
      }
    });
  };
  sfor<NL>([&](auto k) { sfor<NGLL>([&](auto ii) { ub[k][ii] = gb[k][ii] = 0.0; }); });
  auto transverse = [&](auto l) {
    averages(l);
    sfor<NL - 1>([&](auto kt) { next_level(l, kt); });
    sfor<NA - 1>([&](auto km) { flux_rev(l, std::integral_constant<int, NA - 2 - km>{}); });
  };
  transverse(std::integral_constant<int, T1>{});
  transverse(std::integral_constant<int, T2>{});
  averages(std::integral_constant<int, idR>{});
  averages(std::integral_constant<int, NM>{});
  averages(std::integral_constant<int, idT>{});
  if constexpr (DIR == 2) svb = srcb;
  sfor<NA - 1>([&](auto km) {
    constexpr int kt = NA - 2 - km;
    constexpr double rkt1 = 1.0 / (kt + 1.0);
    constexpr bool last = km == 0;
    const double ndt = K.ndt[kt], tav = K.tav[kt + 1];
    if constexpr (!last) {
      sfor<NGLL>([&](auto ii) {
        const double xb = ub[kt + 1][ii] * rr[ii];
        qb[NM][kt + 1][ii] += xb;
        qb[idR][0][ii] = fma(-xb, u[kt + 1][ii], qb[idR][0][ii]);
        sfor<kt + 1>([&](auto j) {
          qb[idR][j + 1][ii] = fma(-xb, u[kt - j][ii], qb[idR][j + 1][ii]);
          ub[kt - j][ii] = fma(-xb, q[idR][j + 1][ii], ub[kt - j][ii]);
        });
        const double Xb = gb[kt + 1][ii] * rrt[ii], tgb = Xb * rkt1;
        qb[idT][0][ii] = fma(-Xb, g[kt + 1][ii], qb[idT][0][ii]);
        // g[0] q[idT][kt+1]: once by itself, once as the sum's first term
        gb[0][ii] = fma((2.0 * GAMMA) * Xb, q[idT][kt + 1][ii], gb[0][ii]);
        qb[idT][kt + 1][ii] = fma((2.0 * GAMMA) * Xb, g[0][ii], qb[idT][kt + 1][ii]);
        sfor<kt>([&](auto im) {
          constexpr int ir = im + 1;
          const double wb = (kt + 1.0 - ir) * tgb;
          gb[ir][ii] = fma(GAMMA * wb, q[idT][kt + 1 - ir][ii], gb[ir][ii]);
          qb[idT][kt + 1 - ir][ii] = fma(GAMMA * wb, g[ir][ii], qb[idT][kt + 1 - ir][ii]);
          qb[idT][ir][ii] = fma(-wb, g[kt + 1 - ir][ii], qb[idT][ir][ii]);
          gb[kt + 1 - ir][ii] = fma(-wb, q[idT][ir][ii], gb[kt + 1 - ir][ii]);
        });
      });
      if constexpr (DIR == 2) {
        if (bg.wall_top) qb[idW][kt + 1][E] = 0.0;
        if (bg.wall_bot) qb[idW][kt + 1][0] = 0.0;
      }
    }
    if constexpr (DIR == 2) {
      // the source: in the momentum's level kt + 1, and in its average
      sfor<NGLL>([&](auto ii) {
        double wb = 0.0;
        if constexpr (!last) wb = qb[idW][kt + 1][ii];
        else if constexpr (ii == 0) wb = tav * lb[idW];
        else if constexpr (ii == E) wb = tav * hb[idW];
        if constexpr (kt == 0) svb += wb;
        else qb[idR][kt][ii] = fma(-GRAV * rkt1, wb, qb[idR][kt][ii]);
      });
      const double s = -GRAV * (tav * ndt) * srcb;
      qb[NM][kt][E] += s;
      qb[NM][kt][0] -= s;
    }
    const std::integral_constant<int, kt> k{};
    flux_rev(std::integral_constant<int, idR>{}, k);
    flux_rev(std::integral_constant<int, NM>{}, k);
    flux_rev(std::integral_constant<int, idT>{}, k);
  });
  // level 0
  if constexpr (DIR == 2) qb[idR][0][E] -= svb * GRAV;
  sfor<NGLL>([&](auto ii) {
    const double xb = ub[0][ii] * rr[ii];
    qb[NM][0][ii] += xb;
    qb[idR][0][ii] = fma(-xb, u[0][ii], qb[idR][0][ii]);
    qb[idT][0][ii] = fma(GAMMA * gb[0][ii], g[0][ii] * rrt[ii], qb[idT][0][ii]);
  });
  if constexpr (DIR == 2) {
    if (bg.wall_top) qb[idW][0][E] = 0.0;
    if (bg.wall_bot) qb[idW][0][0] = 0.0;
  }
  sfor<5>([&](auto l) { sfor<NGLL>([&](auto ii) { q0b[l][ii] = qb[l][0][ii]; }); });
}

// stb += (d (eL, eR, src_avg) / d st)^T (eLb, eRb, srcb) for one cell
template <int ORD, int NGLL, int DIR>
AWFL_HD void cell_adj(const double (&st)[5][ORD], const CellBg<NGLL>& bg, bool weno_s, bool weno_w,
                      const SweepK& K, const double (&eLb)[5], const double (&eRb)[5], double srcb,
                      double (&stb)[5][ORD]) {
  double q0[5][NGLL], q0b[5][NGLL];
  cell_recon<ORD, NGLL>(st, weno_s, weno_w, q0);
  cell_dt_adj<NGLL, DIR>(q0, bg, K, eLb, eRb, srcb, q0b);
  sfor<5>([&](auto l) {
    double ub[ORD];
    sfor<ORD>([&](auto s) { ub[s] = 0.0; });
    reconstruct_adj<ORD, NGLL>(st[l], (l == idR || l == idT) ? weno_s : weno_w, q0b[l], ub);
    sfor<ORD>([&](auto s) { stb[l][s] += ub[s]; });
  });
}

#undef AWFL_HD

}  // namespace adj
}  // namespace awfl
