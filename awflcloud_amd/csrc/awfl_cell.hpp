// awfl_cell.hpp -- per-cell and per-face numerics of one split sweep, in
// registers: WENO reconstruction to GLL points, ADER differential transform
// of the Euler fluxes, time averaging of the cell-edge states, and the
// upwind characteristic Riemann flux.
//
// The values are the reference's formulas', in forms of fewer operations: WENO5 and
// WENO3 in differences of the stencil (reconstruct_w5, reconstruct_w3), the general
// reconstruction with folded maps (weno_coefs), the transform by the normal velocity's
// Taylor coefficients (cell_transform), the flux in differences of the two sides
// (riemann); reciprocals (rcp(), ~1 ulp) for divisions, several from one where they go
// together, and (rho theta)^GAMMA by pow_gamma().  Multiply-adds of the difference
// forms, the transform and the flux are written out (fm) with the compiler's own
// contraction off, so that every kernel rounds them alike; the general reconstruction
// contracts as the compiler chooses.  The reference's operation order is the CPU
// oracle's and, for test builds, awfl_cell_ref.hpp's.
//   WENO ..................... WenoLimiter.h:12-25, 93-172
//   reconstruction ........... Spatial_euler3d_cons_expl_cart_fv_Agrid.h (S:) 1800-1833
//   level-0 products ......... S:704-715, 1067-1078, 1428-1440
//   differential transform ... S:1837-1916 (x), 1920-2000 (y), 2004-2091 (z)
//   time averages ............ S:2130-2177
//   Riemann fluxes ........... S:842-887 (x), 1202-1245 (y), 1583-1629 (z)
#pragma once
#include <type_traits>

#include "awfl_fastmath.hpp"   // HIP runtime, or host stand-ins for __host__/__device__
#include "awfl_tables.hpp"

namespace awfl {

// reciprocal of a positive normal value: refined FP64 (rcp) or the FP32
// hardware estimate (~1 ulp)
__host__ __device__ __forceinline__ double rcp_t(double x) { return rcp(x); }
__host__ __device__ __forceinline__ float rcp_t(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_rcpf(x);
#else
  return 1.0f / x;
#endif
}

// phys_params.h:4-10
constexpr double GRAV = 9.81;
constexpr double C0 = 27.5629410929725921310572974482;
constexpr double GAMMA = 1.40027894002789400278940027894;
constexpr double WENO_EPS = 1.0e-20;     // WenoLimiter.h:22, 100

enum { idR = 0, idU = 1, idV = 2, idW = 3, idT = 4 };

// ---------------------------------------------------------------------------
// truncated total-variation indicator: the generated quadratic form of
// coefs_to_tv<N>, terms summed left to right
// ---------------------------------------------------------------------------
template <int N, int M, class T>
__host__ __device__ __forceinline__ T tv_eval(const T (&a)[M]) {
  // grouped by the first coefficient: sum_j a_j (sum_{terms (j,k)} c a_k)
  T r = 0;
  bool first = true;
  sfor<N>([&](auto j) {
    T inner = 0;
    bool any = false;
    sfor<Tv<N>::n>([&](auto t) {
      if constexpr (Tv<N>::j[t] == j) {
        constexpr T c = (T)Tv<N>::c[t];
        constexpr int k = Tv<N>::k[t];
        inner = any ? inner + c * a[k] : c * a[k];
        any = true;
      }
    });
    if (any) {
      r = first ? a[j] * inner : r + a[j] * inner;
      first = false;
    }
  });
  return r;
}

// ex[i] = prod_{j != i} b[j] and P = prod_j b[j] (prefix/suffix products)
template <int N, class T>
__host__ __device__ __forceinline__ void excl_products(const T (&b)[N], T (&ex)[N], T& P) {
  T pre[N], suf[N];
  pre[0] = 1.0;
  sfor<N - 1>([&](auto i) {
    if constexpr (i == 0) pre[1] = b[0];
    else pre[i + 1] = pre[i] * b[i];
  });
  suf[N - 1] = 1.0;
  sfor<N - 1>([&](auto m) {
    constexpr int i = N - 2 - m;
    if constexpr (i == N - 2) suf[i] = b[N - 1];
    else suf[i] = suf[i + 1] * b[i + 1];
  });
  sfor<N>([&](auto i) {
    if constexpr (i == 0) ex[i] = suf[0];
    else if constexpr (i == N - 1) ex[i] = pre[N - 1];
    else ex[i] = pre[i] * suf[i];
  });
  P = pre[N - 1] * b[N - 1];
}

// The bridge polynomial's coefficients as one linear map of the stencil,
// [cell][coef]: (recon[hs+1] - sum_i idl_i recon[i] on cells i..i+hs) /
// idl[hs+1], the three statements of WenoLimiter.h:117-131 (full-stencil
// polynomial, subtraction of the weighted candidates, scaling) folded into
// one table at compile time; its values differ from theirs by rounding only.
template <int ORD>
struct BridgeMap {
  double m[ORD][ORD];
  constexpr BridgeMap() : m{} {
    using W = Weno<ORD>;
    constexpr int hs = W::hs;
    for (int s = 0; s < ORD; s++)
      for (int ii = 0; ii < ORD; ii++) {
        double t = W::recon[hs + 1][s][ii];
        if (ii <= hs)
          for (int i = 0; i <= hs; i++)
            if (s - i >= 0 && s - i <= hs) t -= W::idl[i] * W::recon[i][s - i][ii];
        m[s][ii] = t * (1.0 / W::idl[hs + 1]);
      }
  }
};
template <int ORD>
inline constexpr BridgeMap<ORD> kBridge{};

// The bridge map is mirror-symmetric: column c (coefficient c) has
// m[hs+k][c] = (-1)^c m[hs-k][c] (odd columns vanish at the centre), so it is
// applied to the sums u[hs+k] + u[hs-k] (even c) or differences (odd c).
// kind[c]: 1 symmetric, -1 antisymmetric, 0 neither (the plain map is used);
// cm[c] the centre entry, cf[c][k] the coefficient of pair k.
template <int ORD>
struct BridgeMirror {
  int kind[ORD];
  double cm[ORD];
  double cf[ORD][ORD];
  constexpr BridgeMirror() : kind(), cm(), cf() {
    constexpr int hs = (ORD - 1) / 2;
    for (int c = 0; c < ORD; c++) {
      double mx = 0.0;
      for (int s = 0; s < ORD; s++) {
        const double v = kBridge<ORD>.m[s][c];
        mx = v > mx ? v : (-v > mx ? -v : mx);
      }
      const double tol = 1e-12 * mx;
      bool sym = true, anti = true;
      for (int k = 1; k <= hs; k++) {
        const double p = kBridge<ORD>.m[hs + k][c], q = kBridge<ORD>.m[hs - k][c];
        const double ds = p - q, da = p + q;
        if (ds > tol || -ds > tol) sym = false;
        if (da > tol || -da > tol) anti = false;
      }
      const double mid = kBridge<ORD>.m[hs][c];
      if (mid > tol || -mid > tol) anti = false;
      kind[c] = sym ? 1 : (anti ? -1 : 0);
      cm[c] = sym ? mid : 0.0;
      for (int k = 1; k <= hs; k++)
        cf[c][k] = sym ? 0.5 * (kBridge<ORD>.m[hs + k][c] + kBridge<ORD>.m[hs - k][c])
                       : 0.5 * (kBridge<ORD>.m[hs + k][c] - kBridge<ORD>.m[hs - k][c]);
    }
  }
};
template <int ORD>
inline constexpr BridgeMirror<ORD> kBridgeMirror{};

// Every candidate polynomial, the full-stencil polynomial and so the bridge
// and any convex combination of them have the centre cell's average over the
// centre cell [-1/2, 1/2]: a0 + sum_{c even >= 2} a_c / ((c + 1) 2^c) = u_hs.
// So a reconstruction's constant coefficient need not be formed: its GLL
// values are u_hs + sum_{c >= 1} (x^c - [c even] / ((c + 1) 2^c)) a_c.  The
// map m[c][ii] holds those coefficients (row 0 unused).
template <int ORD, int NGLL>
struct AvgProjMap {
  double m[ORD][NGLL];
  constexpr AvgProjMap() : m() {
    using P = Proj<ORD, NGLL>;
    for (int c = 0; c < ORD; c++) {
      double k = 0.0;
      if (c % 2 == 0) {
        double p2 = 1.0;
        for (int e = 0; e < c; e++) p2 *= 2.0;
        k = 1.0 / ((c + 1) * p2);
      }
      for (int ii = 0; ii < NGLL; ii++) m[c][ii] = c == 0 ? 0.0 : P::c2g[c][ii] - P::c2g[0][ii] * k;
    }
  }
};
template <int ORD, int NGLL>
inline constexpr AvgProjMap<ORD, NGLL> kAvgProj{};

// ---------------------------------------------------------------------------
// weno::compute_weno_coefs: ord cell averages u -> ord polynomial coefficients
// ---------------------------------------------------------------------------
// NOAVG: the constant coefficients (candidates, bridge and aw[0]) are not
// formed (aw[0] is left unset); see AvgProjMap.
template <int ORD, class T, bool NOAVG = false>
__host__ __device__ __forceinline__ void weno_coefs(const T (&u)[ORD], T (&aw)[ORD]) {
  using W = Weno<ORD>;
  constexpr int hs = W::hs;
  T a[hs + 2][ORD];
  // hs+1 degree-hs candidates on sub-stencils i..i+hs (WenoLimiter.h:110-116)
  sfor<hs + 1>([&](auto i) {
    sfor<hs + 1>([&](auto ii) {
      if constexpr (NOAVG && ii == 0) return;
      T t = -0.0;
      sfor<hs + 1>([&](auto s) {
        constexpr T cf = (T)W::recon[i][s][ii];
        if constexpr (cf != 0) t += cf * u[i + s];
      });
      a[i][ii] = t;
    });
  });
  // "bridge" polynomial (:117-131): the full-stencil polynomial less the
  // weighted candidates, scaled, as one constant map of the stencil
#if AWFL_PARITY & AWFL_PAR_BRIDGE
  sfor<ORD>([&](auto ii) {
    if constexpr (NOAVG && ii == 0) return;
    T t = -0.0;
    sfor<ORD>([&](auto s) { t += (T)W::recon[hs + 1][s][ii] * u[s]; });
    if constexpr (ii <= hs) sfor<hs + 1>([&](auto i) { t -= (T)W::idl[i] * a[i][ii]; });
    a[hs + 1][ii] = t / (T)W::idl[hs + 1];
  });
#else
  T usum[hs + 1], udif[hs + 1];
  sfor<hs>([&](auto km) {
    constexpr int k = km + 1;
    usum[k] = u[hs + k] + u[hs - k];
    udif[k] = u[hs + k] - u[hs - k];
  });
  sfor<ORD>([&](auto ii) {
    if constexpr (NOAVG && ii == 0) return;
    T t = -0.0;
    if constexpr (kBridgeMirror<ORD>.kind[ii] == 1) {
      if constexpr (kBridgeMirror<ORD>.cm[ii] != 0) t = (T)kBridgeMirror<ORD>.cm[ii] * u[hs];
      sfor<hs>([&](auto km) {
        constexpr T cf = (T)kBridgeMirror<ORD>.cf[ii][km + 1];
        if constexpr (cf != 0) t += cf * usum[km + 1];
      });
    } else if constexpr (kBridgeMirror<ORD>.kind[ii] == -1) {
      sfor<hs>([&](auto km) {
        constexpr T cf = (T)kBridgeMirror<ORD>.cf[ii][km + 1];
        if constexpr (cf != 0) t += cf * udif[km + 1];
      });
    } else {
      sfor<ORD>([&](auto s) {
        constexpr T cf = (T)kBridge<ORD>.m[s][ii];
        if constexpr (cf != 0) t += cf * u[s];
      });
    }
    a[hs + 1][ii] = t;
  });
#endif
  // total variation of every candidate (:133-143), sigma blend (:145-151)
  T tv[hs + 2];
  sfor<hs + 1>([&](auto i) { tv[i] = tv_eval<hs + 1>(a[i]); });
  tv[hs + 1] = tv_eval<ORD>(a[hs + 1]);
  T lo_avg = 0;
  sfor<hs + 1>([&](auto i) { lo_avg += tv[i]; });
  lo_avg *= (T)(1.0 / (hs + 1));
  constexpr T sigma = (T)W::sigma;
  tv[hs + 1] = lo_avg + (tv[hs + 1] - lo_avg) * sigma;
  // weights ~ idl / TV^2, convexify, map, convexify (:153-161).  Each
  // normalisation w_i = (a_i / b_i) / (sum_k a_k / b_k + eps) is formed over
  // the common denominator: a_i prod_{j!=i} b_j / (sum_k a_k prod_{j!=k} b_j
  // + eps prod_j b_j), one reciprocal instead of hs+3 divisions.
  T w[hs + 2];
  if constexpr (std::is_same<T, double>::value) {
    {
      T D[hs + 2], ex[hs + 2], P;
      sfor<hs + 2>([&](auto i) { D[i] = tv[i] * tv[i] + WENO_EPS; });
      excl_products<hs + 2>(D, ex, P);
      T N = 0.0;
      sfor<hs + 2>([&](auto i) {
        constexpr double d = W::idl[i];
        w[i] = d * ex[i];
        N += w[i];
      });
      T rs = rcp(fma(WENO_EPS, P, N));
      sfor<hs + 2>([&](auto i) { w[i] *= rs; });
    }
    {
      T A[hs + 2], E[hs + 2], ex[hs + 2], P;
      sfor<hs + 2>([&](auto i) {
        constexpr double d = W::idl[i];
        A[i] = w[i] * (d + d * d - 3.0 * d * w[i] + w[i] * w[i]);
        E[i] = d * d + w[i] * (1.0 - 2.0 * d);
      });
      excl_products<hs + 2>(E, ex, P);
      T M = 0.0;
      sfor<hs + 2>([&](auto i) {
        w[i] = A[i] * ex[i];
        M += w[i];
      });
      T rs = rcp(fma(WENO_EPS, P, M));
      sfor<hs + 2>([&](auto i) { w[i] *= rs; });
    }
  } else {
    // the tangent-linear scalar: one reciprocal per weight and the map as
    // written, the statements the hand-written reverse follows
    sfor<hs + 2>([&](auto i) {
      constexpr T d = (T)W::idl[i];
      w[i] = d * rcp_t(tv[i] * tv[i] + (T)WENO_EPS);
    });
    T sum = 0;
    sfor<hs + 2>([&](auto i) { sum += w[i]; });
    T rs = rcp_t(sum + (T)WENO_EPS);
    sfor<hs + 2>([&](auto i) { w[i] *= rs; });
    sfor<hs + 2>([&](auto i) {
      constexpr T d = (T)W::idl[i];
      w[i] = w[i] * (d + d * d - (T)3 * d * w[i] + w[i] * w[i]) * rcp_t(d * d + w[i] * ((T)1 - (T)2 * d));
    });
    sum = 0;
    sfor<hs + 2>([&](auto i) { sum += w[i]; });
    rs = rcp_t(sum + (T)WENO_EPS);
    sfor<hs + 2>([&](auto i) { w[i] *= rs; });
  }
  // weighted sum (:163-171); candidates have no coefficients above hs
  sfor<ORD>([&](auto ii) {
    if constexpr (NOAVG && ii == 0) return;
    T t = -0.0;
    sfor<hs + 2>([&](auto i) {
      if constexpr (i == hs + 1 || ii <= hs) t += w[i] * a[i][ii];
    });
    aw[ii] = t;
  });
}

// ---------------------------------------------------------------------------
// WENO5 to three GLL points in difference form
// ---------------------------------------------------------------------------
// Everything WENO5 needs of its stencil is a function of the first
// differences d_k = u_{k+1} - u_k.  With the second differences s_i = d_{i+1}
// - d_i, candidate i is u_2 + ... with doubled coefficients 2 a1 = A_i, 2 a2 =
// s_i:  A_0 = 2 d_1 + s_0, A_1 = d_1 + d_2, A_2 = 2 d_2 - s_2.  The full
// polynomial adds only the third and fourth differences M = s_2 - s_0 and Q =
// s_0 - 2 s_1 + s_2, and so does the bridge (it has candidate 1's part with
// weight one: idl_0 = idl_2 and the ideal weights sum to one):
//   2 b1 = A_1 + g2 M, 2 b2 = s_1 - b2 Q, 2 b3 = k3 M, 2 b4 = k4 Q.
// The truncated-TV form of the bridge is then candidate 1's plus M (m1 A_1 +
// mm M) + Q (q1 s_1 + qq Q).  All TVs are carried times four (doubled
// coefficients), which the weights, homogeneous in them, do not see; eps is
// scaled with them.  106 FP64 operations against 137 for the general form
// with folded maps (weno_coefs + projection), and the values of smooth fields
// are differenced once, up front, instead of in every map.  The sweeps are
// bound by FP64 issue: a step at 256x256x128 went from 1.258 to 1.148 ms, the
// FP32 form at 512x512x256 from 5.27 to 4.80 ms.
struct Weno5Consts {
  double tvs;                    // 13/3: weight of s^2 in 4 TV of a candidate
  double k0, k1;                 // blended bridge TV: weights of t_0 + t_2 and of t_1
  double m1, mm, q1, qq;         // ... of M A_1, M^2, Q s_1, Q^2
  double c1, c3;                 // ideal weights over idl_0
  double eps, epsn;              // eps for (4 TV)^2, and of the first normalisation
  double od_m, ev_q, md_q;       // odd part: M; even parts at the edges and the centre: Q
  constexpr Weno5Consts() : tvs(), k0(), k1(), m1(), mm(), q1(), qq(), c1(), c3(), eps(), epsn(), od_m(), ev_q(), md_q() {
    using W = Weno<5>;
    double lo2 = 0, c11 = 0, c13 = 0, c22 = 0, c24 = 0, c33 = 0, c44 = 0;
    for (int t = 0; t < Tv<3>::n; t++)
      if (Tv<3>::j[t] == 2 && Tv<3>::k[t] == 2) lo2 = Tv<3>::c[t];
    for (int t = 0; t < Tv<5>::n; t++) {
      const int j = Tv<5>::j[t], k = Tv<5>::k[t];
      const double c = Tv<5>::c[t];
      if (j == 1 && k == 1) c11 = c;
      if (j == 1 && k == 3) c13 = c;
      if (j == 2 && k == 2) c22 = c;
      if (j == 2 && k == 4) c24 = c;
      if (j == 3 && k == 3) c33 = c;
      if (j == 4 && k == 4) c44 = c;
    }
    const double i0 = W::idl[0], i3 = W::idl[3], sg = W::sigma;
    const double g2 = (i0 - 5.0 / 24.0) / i3, b2 = (i0 + 0.125) / i3, k3 = 1.0 / (6.0 * i3), k4 = 1.0 / (12.0 * i3);
    tvs = lo2;
    k0 = (1.0 - sg) / 3.0;
    k1 = k0 + sg;
    m1 = sg * (2.0 * c11 * g2 + c13 * k3);
    mm = sg * (c11 * g2 * g2 + c13 * k3 * g2 + c33 * k3 * k3);
    q1 = sg * (c24 * k4 - 2.0 * c22 * b2);
    qq = sg * (c22 * b2 * b2 - c24 * k4 * b2 + c44 * k4 * k4);
    c1 = W::idl[1] / i0;
    c3 = i3 / i0;
    eps = 16.0 * WENO_EPS;
    epsn = WENO_EPS / (16.0 * i0);
    od_m = g2 + 0.25 * k3;
    ev_q = k4 / 40.0 - b2 / 12.0;
    md_q = b2 / 24.0 - k4 / 160.0;
  }
};
inline constexpr Weno5Consts kW5{};

// one FP32 reciprocal per weight, or the FP64 common denominator: w_i ~ c_i /
// D_i (c_0 = c_2 = 1), normalised with eps (WenoLimiter.h:153-156)
template <class T>
__host__ __device__ __forceinline__ void weno5_first_weights(const T (&D)[4], T (&w)[4]) {
  AWFL_NO_CONTRACT
  constexpr T c1 = (T)kW5.c1, c3 = (T)kW5.c3;
  if constexpr (std::is_same<T, double>::value) {
    const T D01 = D[0] * D[1], D23 = D[2] * D[3];
    const T n0 = D[1] * D23, n1 = (D[0] * D23) * c1, n2 = D01 * D[3], n3 = (D01 * D[2]) * c3;
    const T rs = rcp(fm((T)kW5.epsn, D01 * D23, (n0 + n1) + (n2 + n3)));
    w[0] = n0 * rs;
    w[1] = n1 * rs;
    w[2] = n2 * rs;
    w[3] = n3 * rs;
  } else {
    const T n0 = rcp_t(D[0]), n1 = c1 * rcp_t(D[1]), n2 = rcp_t(D[2]), n3 = c3 * rcp_t(D[3]);
    const T rs = rcp_t(((n0 + n1) + (n2 + n3)) + (T)kW5.epsn);
    w[0] = n0 * rs;
    w[1] = n1 * rs;
    w[2] = n2 * rs;
    w[3] = n3 * rs;
  }
}

// map_weights' numerator and denominator (WenoLimiter.h:12-18): w (d + d^2 - 3
// d w + w^2) / (d^2 + w (1 - 2 d))
template <int I, int ORD, class T>
__host__ __device__ __forceinline__ void weno_map(T w, T& A, T& E) {
  constexpr double d = Weno<ORD>::idl[I];
  constexpr T d3 = (T)(-3.0 * d), dd = (T)(d + d * d), d2 = (T)(d * d), e1 = (T)(1.0 - 2.0 * d);
  A = w * fm(w, w + d3, dd);
  E = fm(w, e1, d2);
}

template <class T>
__host__ __device__ __forceinline__ void reconstruct_w5(const T (&u)[5], T (&g)[3]) {
  AWFL_NO_CONTRACT
  const T d0 = u[1] - u[0], d1 = u[2] - u[1], d2 = u[3] - u[2], d3 = u[4] - u[3];
  const T s0 = d1 - d0, s1 = d2 - d1, s2 = d3 - d2;
  const T A0 = fm((T)2, d1, s0), A1 = d1 + d2, A2 = fm((T)2, d2, -s2);
  const T M = s2 - s0, Q = fm((T)-2, s1, s0 + s2);
  // total variation (times four) of the candidates and, blended with their
  // average by sigma, of the bridge (WenoLimiter.h:133-151)
  const T t0 = fm((T)kW5.tvs * s0, s0, A0 * A0);
  const T t1 = fm((T)kW5.tvs * s1, s1, A1 * A1);
  const T t2 = fm((T)kW5.tvs * s2, s2, A2 * A2);
  T th = fm((T)kW5.k1, t1, (T)kW5.k0 * (t0 + t2));
  th = fm(M, fm((T)kW5.m1, A1, (T)kW5.mm * M), th);
  th = fm(Q, fm((T)kW5.q1, s1, (T)kW5.qq * Q), th);
  const T D[4] = {fm(t0, t0, (T)kW5.eps), fm(t1, t1, (T)kW5.eps), fm(t2, t2, (T)kW5.eps), fm(th, th, (T)kW5.eps)};
  T w[4], a[4], e[4];
  weno5_first_weights(D, w);
  weno_map<0, 5>(w[0], a[0], e[0]);
  weno_map<1, 5>(w[1], a[1], e[1]);
  weno_map<2, 5>(w[2], a[2], e[2]);
  weno_map<3, 5>(w[3], a[3], e[3]);
  // second normalisation over the common denominator; its sum is of order one
  // times prod e, so that eps (1e-20) vanishes in it.  rs is applied to the sums.
  const T e01 = e[0] * e[1], e23 = e[2] * e[3];
  const T W0 = a[0] * (e[1] * e23), W1 = a[1] * (e[0] * e23), W2 = a[2] * (e01 * e[3]), W3 = a[3] * (e01 * e[2]);
  const T W13 = W1 + W3;
  const T rs = rcp_t((W0 + W2) + W13);
  const T w3 = W3 * rs, wM = w3 * M, wQ = w3 * Q;
  // od: four times the odd part at x = 1/2; ev: twelve times the even part
  const T od = fm(rs, fm(W2, A2, fm(W13, A1, W0 * A0)), (T)kW5.od_m * wM);
  const T ev = rs * fm(W2, s2, fm(W13, s1, W0 * s0));
  const T end = u[2] + fm(ev, (T)(1.0 / 12.0), (T)kW5.ev_q * wQ);
  g[0] = fm((T)-0.25, od, end);
  g[1] = u[2] + fm(ev, (T)(-1.0 / 24.0), (T)kW5.md_q * wQ);
  g[2] = fm((T)0.25, od, end);
}

// ---------------------------------------------------------------------------
// WENO3 to two GLL points in difference form: candidates d_0 and d_1 (their
// slopes), bridge slope (d_0 + d_1)/2 and curvature k2 (d_1 - d_0)/2
// ---------------------------------------------------------------------------
struct Weno3Consts {
  double k0, ks, kd;             // blended bridge TV: t_0 + t_1, (d0 + d1)^2, (d1 - d0)^2
  double c2, epsn, ev;           // ideal weight over idl_0, eps of the first normalisation, even part
  constexpr Weno3Consts() : k0(), ks(), kd(), c2(), epsn(), ev() {
    using W = Weno<3>;
    double c11 = 0, c22 = 0;
    for (int t = 0; t < Tv<3>::n; t++) {
      if (Tv<3>::j[t] == 1 && Tv<3>::k[t] == 1) c11 = Tv<3>::c[t];
      if (Tv<3>::j[t] == 2 && Tv<3>::k[t] == 2) c22 = Tv<3>::c[t];
    }
    const double i0 = W::idl[0], i2 = W::idl[2], sg = W::sigma, k2 = 1.0 / i2;
    k0 = (1.0 - sg) / 2.0;
    ks = sg * c11 / 4.0;
    kd = sg * c22 * k2 * k2 / 4.0;
    c2 = i2 / i0;
    epsn = WENO_EPS / i0;
    ev = k2 / 12.0;
  }
};
inline constexpr Weno3Consts kW3{};

template <class T>
__host__ __device__ __forceinline__ void reconstruct_w3(const T (&u)[3], T (&g)[2]) {
  AWFL_NO_CONTRACT
  const T d0 = u[1] - u[0], d1 = u[2] - u[1];
  const T S = d0 + d1, Q = d1 - d0;
  const T t0 = d0 * d0, t1 = d1 * d1;
  const T th = fm((T)kW3.kd * Q, Q, fm((T)kW3.ks * S, S, (T)kW3.k0 * (t0 + t1)));
  const T D[3] = {fm(t0, t0, (T)WENO_EPS), fm(t1, t1, (T)WENO_EPS), fm(th, th, (T)WENO_EPS)};
  T w[3], a[3], e[3];
  if constexpr (std::is_same<T, double>::value) {
    const T D01 = D[0] * D[1];
    const T n0 = D[1] * D[2], n1 = D[0] * D[2], n2 = (T)kW3.c2 * D01;
    const T rs = rcp(fm((T)kW3.epsn, D01 * D[2], (n0 + n1) + n2));
    w[0] = n0 * rs;
    w[1] = n1 * rs;
    w[2] = n2 * rs;
  } else {
    const T n0 = rcp_t(D[0]), n1 = rcp_t(D[1]), n2 = (T)kW3.c2 * rcp_t(D[2]);
    const T rs = rcp_t(((n0 + n1) + n2) + (T)kW3.epsn);
    w[0] = n0 * rs;
    w[1] = n1 * rs;
    w[2] = n2 * rs;
  }
  weno_map<0, 3>(w[0], a[0], e[0]);
  weno_map<1, 3>(w[1], a[1], e[1]);
  weno_map<2, 3>(w[2], a[2], e[2]);
  const T W0 = a[0] * (e[1] * e[2]), W1 = a[1] * (e[0] * e[2]), W2 = a[2] * (e[0] * e[1]);
  const T rs = rcp_t((W0 + W1) + W2);
  const T hw = (T)0.5 * W2;
  const T od = ((T)0.5 * rs) * fm(W0 + hw, d0, (W1 + hw) * d1);
  const T mid = fm((T)kW3.ev, (W2 * rs) * Q, u[1]);
  g[0] = mid - od;
  g[1] = mid + od;
}

// reconstruct_gll_values (S:1800-1833): ord stencil -> NGLL point values
template <int ORD, int NGLL, class T>
__host__ __device__ __forceinline__ void reconstruct(const T (&u)[ORD], bool doweno, T (&g)[NGLL]) {
  using P = Proj<ORD, NGLL>;
  // the difference forms serve the sweeps' scalars (double and float); the
  // tangent-linear scalar keeps the general form, and the bridge parity build
  // the reference's three statements
  constexpr bool diff = (std::is_same<T, double>::value || std::is_same<T, float>::value) &&
                        !(AWFL_PARITY & AWFL_PAR_BRIDGE);
  if (doweno) {
    if constexpr (diff && ORD == 5 && NGLL == 3) {
      reconstruct_w5(u, g);
      return;
    } else if constexpr (diff && ORD == 3 && NGLL == 2) {
      reconstruct_w3(u, g);
      return;
    }
    // the weighted polynomial's GLL values from the centre cell's average and
    // its non-constant coefficients (AvgProjMap; c2g[0][.] = 1)
    T aw[ORD];
    weno_coefs<ORD, T, true>(u, aw);
    sfor<NGLL>([&](auto ii) {
      T t = u[(ORD - 1) / 2];
      sfor<ORD>([&](auto s) {
        if constexpr (s > 0) {
          constexpr T cf = (T)kAvgProj<ORD, NGLL>.m[s][ii];
          if constexpr (cf != 0) t += cf * aw[s];
        }
      });
      g[ii] = t;
    });
  } else {
    sfor<NGLL>([&](auto ii) {
      T t = -0.0;
      sfor<ORD>([&](auto s) {
        constexpr T cf = (T)P::s2g[s][ii];
        if constexpr (cf != 0) t += cf * u[s];
      });
      g[ii] = t;
    });
  }
}

// Background seen by one cell of a sweep.  X and Y add the cell averages
// hyDensCells/hyDensThetaCells (S:680, 697, 1043, 1060); Z adds the GLL point
// values and subtracts the background pressure (S:1400, 1421, 2042).
// Each background rho*theta value B also comes with B^GAMMA as a double-double
// (h, l) and 1/B, the reference point of pow_gamma_near.
struct PowRef {
  double h, l, rb, b;
};

template <int NGLL>
struct CellBg {
  double r, rt;            // x/y: cell averages of the background
  PowRef pt;               // x/y: power reference of rt
  double rG[NGLL];         // z: hyDensGLL(k, :)
  double rtG[NGLL];        // z: hyDensThetaGLL(k, :)
  double pG[NGLL];         // z: hyPressureGLL(k, :)
  PowRef ptG[NGLL];        // z: power references of rtG
  bool wall_bot, wall_top; // z: solid wall and k == 0 / k == nz-1
};

// power references of a face: for (r t) of the averaged state and for the
// recomposed q5 of the Riemann flux
struct FaceRef {
  PowRef rt, q5;
};

// Launch constants of one sweep: dt, 1/d along the sweep, the differential
// transform factors -1/(d (kt+1)) and the time-average weights dt^kt/(kt+1).
constexpr int KMAX = 9;
struct SweepK {
  double dt;
  double rd;              // 1 / dsw
  double ndt[KMAX];       // -1 / (dsw (kt+1)), kt = 0..NA-2
  double tav[KMAX];       // dt^kt / (kt+1), kt = 1..NA-1 (tav[0] unused)
  double dsw;             // grid spacing along the sweep (reference-order parity builds)
  unsigned char* br;      // upwind branch per face (record / replay kernels only)
};

// ---------------------------------------------------------------------------
// n times the derivative of the point values F along the cell at its GLL
// points (Deriv<NGLL>, the collocation derivative).  With two and three
// points it is formed from F's first and second difference.
// ---------------------------------------------------------------------------
template <int NGLL>
__host__ __device__ __forceinline__ void gll_deriv(const double (&F)[NGLL], double n, double (&d)[NGLL]) {
  AWFL_NO_CONTRACT
  if constexpr (NGLL == 2) {
    d[0] = d[1] = (F[1] - F[0]) * n;
  } else if constexpr (NGLL == 3) {
    const double a = (F[2] - F[0]) * n, c = fm(-2.0, F[1], F[0] + F[2]), h = 2.0 * n;
    d[0] = fm(-h, c, a);
    d[1] = a;
    d[2] = fm(h, c, a);
  } else {
    sfor<NGLL>([&](auto ii) {
      double t = -0.0;
      sfor<NGLL>([&](auto s) {
        constexpr double D = Deriv<NGLL>::m[s][ii];
        if constexpr (D != 0.0) t = fm(D, F[s], t);
      });
      d[ii] = t * n;
    });
  }
}

// eL, eR += n times that derivative at the cell's two edges
template <int NGLL>
__host__ __device__ __forceinline__ void gll_deriv_edges(const double (&F)[NGLL], double n, double& eL, double& eR) {
  AWFL_NO_CONTRACT
  if constexpr (NGLL == 3) {
    const double a = F[2] - F[0], c = fm(-2.0, F[1], F[0] + F[2]), h = 2.0 * n;
    eL = fm(-h, c, fm(n, a, eL));
    eR = fm(h, c, fm(n, a, eR));
  } else {
    double d[NGLL];
    gll_deriv<NGLL>(F, n, d);
    eL += d[0];
    eR += d[NGLL - 1];
  }
}

// ---------------------------------------------------------------------------
// One cell of a DIR sweep (0 x, 1 y, 2 z): stencils of the 5 state variables
// along the sweep axis -> time-averaged left/right edge states (and, for z,
// the time- and cell-averaged gravity source of rho*w).
//
// The transform carries the normal velocity's Taylor coefficients u_k: with
// u r = q_nm, u_k = (q_nm,k - sum_{j>=1} r_j u_{k-j}) / r_0, the flux of every
// variable is f_k = sum_j u_j q_{k-j}: the same coefficients as the
// reference's f_k = (sum_j q_nm,j q_{k-j} - sum_{j>=1} r_j f_{k-j}) / r_0,
// with one division per point instead of one per variable and half the
// products.  The last level enters the edge states alone and is formed there.
// The cell average of the z source follows from the quadrature being exact
// for a derivative: sum_s w_s dF/dx(s) = F(last) - F(first).  The sweeps are
// bound by FP64 issue: with gll_deriv, one reciprocal for 1/r and 1/(r t), one
// branch for the cell's powers and riemann()'s difference form, a (5, 3) y
// sweep's cell and face went from 1,020 to 830 FP64 operations and a step at
// 256x256x128 from 1.148 to 1.000 ms; the errors against 64-bit torch did not
// grow (7.6e-15 -> 7.4e-15 of the state).
// ---------------------------------------------------------------------------
// levels(r0, u) receives the density at the GLL points (background added) and
// the normal velocity's Taylor coefficients u[level][point], levels 0 ..
// NGLL-2, which the tracer sweeps' transform takes (S:757-758).
template <int NGLL, int DIR, class Levels>
__host__ __device__ __forceinline__ void cell_transform(const double (&q0)[5][NGLL], const CellBg<NGLL>& bg,
                                               const SweepK& K, double (&eL)[5], double (&eR)[5], double& src_avg,
                                               Levels&& levels) {
  AWFL_NO_CONTRACT
  constexpr int NA = NGLL;             // nAder = ngll (Temporal_ader.h:8)
  constexpr int NM = 1 + DIR;          // momentum normal to the sweep
  static_assert(NA >= 2, "at least one transform level");
  double q[5][NA][NGLL];               // r, ru, rv, rw, rt at levels 0 .. NA-2
  double u[NA][NGLL];                  // normal velocity
  double g[NA][NGLL];                  // (r t)^gamma, levels >= 1 carried doubled (S:1904-1915)
  double rr[NGLL], rrt[NGLL];          // 1/r and 1/(r t) at level 0

  // level 0: the reconstruction, and the background
  sfor<5>([&](auto l) { sfor<NGLL>([&](auto ii) { q[l][0][ii] = q0[l][ii]; }); });
  // S:1439 assigns a scalar to the whole SArray: every entry of the source's
  // level 0 holds the value of the last GLL point
  const double sv = DIR == 2 ? -GRAV * q[idR][0][NGLL - 1] : 0.0;
  // (r t)^gamma: r t = rho*theta up to an ulp.  The series near the
  // background runs for every lane; the general power replaces it where a
  // point is further off.
  bool near = true;
  sfor<NGLL>([&](auto ii) {
    const PowRef& pr = DIR == 2 ? bg.ptG[ii] : bg.pt;
    const double e = q[idT][0][ii] * pr.rb;
    g[0][ii] = pow_gamma_series(e, pr.h, pr.l);
    near = near & (fabs(e) <= NEAR_MAX);
    if constexpr (DIR == 2) {
      q[idR][0][ii] += bg.rG[ii];
      q[idT][0][ii] += bg.rtG[ii];
    } else {
      q[idR][0][ii] += bg.r;
      q[idT][0][ii] += bg.rt;
    }
  });
  if (AWFL_PARITY & AWFL_PAR_POW ? true : !near)
    sfor<NGLL>([&](auto ii) {
      const double e = (q[idT][0][ii] - (DIR == 2 ? bg.rtG[ii] : bg.rt)) * (DIR == 2 ? bg.ptG[ii] : bg.pt).rb;
      if (AWFL_PARITY & AWFL_PAR_POW ? true : !(fabs(e) <= NEAR_MAX)) g[0][ii] = pow_gamma_far(q[idT][0][ii]);
    });
  if constexpr (DIR == 2) {            // S:1413-1416
    if (bg.wall_top) q[idW][0][NGLL - 1] = 0.0;
    if (bg.wall_bot) q[idW][0][0] = 0.0;
  }
  sfor<NGLL>([&](auto ii) {
    const double r = q[idR][0][ii], rt = q[idT][0][ii];
    if constexpr (NA > 2) {
      const double z = rcp(r * rt);
      rr[ii] = rt * z;
      rrt[ii] = r * z;
    } else {
      rr[ii] = rcp(r);
    }
    u[0][ii] = q[NM][0][ii] * rr[ii];
  });
  sfor<5>([&](auto l) {
    eL[l] = q[l][0][0];
    eR[l] = q[l][0][NGLL - 1];
  });
  double sa = sv;

  // differential transform: levels 1..NA-1
  sfor<NA - 1>([&](auto kt) {
    constexpr double rkt1 = 1.0 / (kt + 1.0);
    constexpr bool last = kt + 2 == NA;
    const double ndt = K.ndt[kt], tav = K.tav[kt + 1];
    if constexpr (DIR == 2) sa = fm(-GRAV * (tav * ndt), q[NM][kt][NGLL - 1] - q[NM][kt][0], sa);
    sfor<5>([&](auto l) {
      double F[NGLL];
      sfor<NGLL>([&](auto s) {
        if constexpr (l == idR) {
          F[s] = q[NM][kt][s];
        } else {
          double t;
          if constexpr (l == NM) {
            if constexpr (kt == 0) t = DIR == 2 ? fm(C0, g[kt][s], -bg.pG[s]) : C0 * g[kt][s];
            else t = (0.5 * C0) * g[kt][s];
            t = fm(u[0][s], q[l][kt][s], t);
          } else {
            t = u[0][s] * q[l][kt][s];
          }
          sfor<kt>([&](auto j) { t = fm(u[j + 1][s], q[l][kt - 1 - j][s], t); });
          F[s] = t;
        }
      });
      if constexpr (last) {
        gll_deriv_edges<NGLL>(F, ndt * tav, eL[l], eR[l]);
        if constexpr (DIR == 2 && l == idW) {     // the source at level kt, S:2049
          eL[l] = kt == 0 ? fm(tav, sv, eL[l]) : fm((-GRAV * rkt1) * tav, q[idR][kt][0], eL[l]);
          eR[l] = kt == 0 ? fm(tav, sv, eR[l]) : fm((-GRAV * rkt1) * tav, q[idR][kt][NGLL - 1], eR[l]);
        }
      } else {
        double d[NGLL];
        gll_deriv<NGLL>(F, ndt, d);
        sfor<NGLL>([&](auto ii) {
          if constexpr (DIR == 2 && l == idW) d[ii] = kt == 0 ? d[ii] + sv : fm(-GRAV * rkt1, q[idR][kt][ii], d[ii]);
          q[l][kt + 1][ii] = d[ii];
        });
        if constexpr (DIR == 2 && l == idW) {     // S:2051-2055
          if (bg.wall_top) q[idW][kt + 1][NGLL - 1] = 0.0;
          if (bg.wall_bot) q[idW][kt + 1][0] = 0.0;
        }
        eL[l] = fm(q[l][kt + 1][0], tav, eL[l]);   // time averages of the edge values (S:2142-2177)
        eR[l] = fm(q[l][kt + 1][NGLL - 1], tav, eR[l]);
      }
    });
    if constexpr (!last) {
      sfor<NGLL>([&](auto ii) {
        double t = q[NM][kt + 1][ii];
        sfor<kt + 1>([&](auto j) { t = fm(-q[idR][j + 1][ii], u[kt - j][ii], t); });
        u[kt + 1][ii] = t * rr[ii];
        if constexpr (kt == 0) {
          g[1][ii] = (2.0 * GAMMA) * ((g[0][ii] * rrt[ii]) * q[idT][1][ii]);
        } else {
          double tg = 0.0;
          sfor<kt + 1>([&](auto ir) {
            constexpr double wgt = kt + 1.0 - ir;
            double p = (GAMMA * g[ir][ii]) * q[idT][kt + 1 - ir][ii];
            if constexpr (ir > 0) p = fm(-q[idT][ir][ii], g[kt + 1 - ir][ii], p);
            tg = fm(wgt, p, tg);
          });
          g[kt + 1][ii] = fm(GAMMA * g[0][ii], q[idT][kt + 1][ii], tg * rkt1) * rrt[ii];
        }
      });
    }
  });
  if constexpr (DIR == 2) {
    if (bg.wall_top) eR[idW] = 0.0;
    if (bg.wall_bot) eL[idW] = 0.0;
  }

  const double(&r0)[NGLL] = q[idR][0];
  levels(r0, u);
  src_avg = DIR == 2 ? sa : 0.0;       // S:1462, 1489-1492
}

// Reconstruction and transform of a cell.  load_bg() returns the cell's
// background; it is called after the reconstructions, so that a background
// that differs between lanes is not held in registers through them.
template <int ORD, int NGLL, int DIR, class LoadBg, class Levels>
__host__ __device__ __forceinline__ void cell_edges_of(const double (&st)[5][ORD], LoadBg&& load_bg, bool weno_s,
                                              bool weno_w, const SweepK& K, double (&eL)[5], double (&eR)[5],
                                              double& src_avg, Levels&& levels) {
  double q0[5][NGLL];
  sfor<5>([&](auto l) { reconstruct<ORD, NGLL>(st[l], (l == idR || l == idT) ? weno_s : weno_w, q0[l]); });
  const CellBg<NGLL> bg = load_bg();
  cell_transform<NGLL, DIR>(q0, bg, K, eL, eR, src_avg, levels);
}
template <int ORD, int NGLL, int DIR, class Levels>
__host__ __device__ __forceinline__ void cell_edges(const double (&st)[5][ORD], const CellBg<NGLL>& bg, bool weno_s,
                                           bool weno_w, const SweepK& K, double (&eL)[5], double (&eR)[5],
                                           double& src_avg, Levels&& levels) {
  cell_edges_of<ORD, NGLL, DIR>(st, [&]() { return bg; }, weno_s, weno_w, K, eL, eR, src_avg, levels);
}
template <int ORD, int NGLL, int DIR>
__host__ __device__ __forceinline__ void cell_edges(const double (&st)[5][ORD], const CellBg<NGLL>& bg, bool weno_s,
                                           bool weno_w, const SweepK& K, double (&eL)[5], double (&eR)[5],
                                           double& src_avg) {
  cell_edges<ORD, NGLL, DIR>(st, bg, weno_s, weno_w, K, eL, eR, src_avg, [](const auto&, const auto&) {});
}

// ---------------------------------------------------------------------------
// Upwind characteristic flux at one face.  X and Z average primitive
// variables; Y averages the conservative variables (S:1210-1214).  The
// normal velocity test is strict (u > 0).
// ---------------------------------------------------------------------------
// Averages of the two edge states at a face and the reciprocals that go with
// them.  In x and z the velocities and theta are averaged: with X_l = L_l R_0 +
// R_l L_0 they are X_l / (2 L_0 R_0), and 1/r, 1/(L_0 R_0) and 1/t come from
// one reciprocal (of r L_0 R_0 X_4) by products.  The adjoint forms its
// averages here too, so that both take the same upwind side.
struct FaceAvg {
  double r, un, ut1, ut2, t;
  double ir, hit;                      // 1/r, 1/(2 t)
  double iLR;                          // 1/(L_0 R_0) (x and z)
};
template <int DIR>
__host__ __device__ __forceinline__ FaceAvg face_averages(const double (&L)[5], const double (&R)[5]) {
  AWFL_NO_CONTRACT
  constexpr int NM = 1 + DIR;
  // tangential momentum indices in the order the reference uses them
  constexpr int T1 = DIR == 0 ? 2 : 1;
  constexpr int T2 = DIR == 2 ? 2 : 3;
  FaceAvg a;
  a.r = 0.5 * (L[0] + R[0]);
  if constexpr (DIR == 1) {
    a.un = 0.5 * (L[NM] + R[NM]);
    a.ut1 = 0.5 * (L[T1] + R[T1]);
    a.ut2 = 0.5 * (L[T2] + R[T2]);
    a.t = 0.5 * (L[4] + R[4]);
    const double z = rcp(a.r * a.t);
    a.ir = a.t * z;
    a.hit = (0.5 * a.r) * z;
    a.iLR = 0.0;
  } else {
    const double LR = L[0] * R[0];
    const double x4 = fm(L[4], R[0], R[4] * L[0]);
    const double y = LR * x4, z = rcp(y * a.r), iy = z * a.r;
    a.ir = z * y;
    a.iLR = iy * x4;
    a.hit = LR * (iy * LR);
    const double h = 0.5 * a.iLR;
    a.un = fm(L[NM], R[0], R[NM] * L[0]) * h;
    a.ut1 = fm(L[T1], R[0], R[T1] * L[0]) * h;
    a.ut2 = fm(L[T2], R[0], R[T2] * L[0]) * h;
    a.t = x4 * h;
  }
  return a;
}

// un_out receives the averaged normal velocity the flux upwinds with (the
// tracer fluxes upwind with the same value, S:891-900).  With FORCE the
// upwind side of waves 1-3 is up_forced (true: left) instead of the sign
// test: the flux with a frozen branch, for difference checks of the adjoint.
//
// The waves and the recomposed state (S:866-882) are taken together, in
// differences of the two sides, so that 1/t and cs act on differences only:
// with D = (u_n (R_0 - L_0) + L_n - R_n) / (2 cs) and d = (R_4 - L_4) / (2 t),
//   q5 = (L_4 + R_4)/2 + t D,  v = D + d (left upwind) or D - d,
//   q1 = U_0 + v,  q_t = U_t + u_t v  (U the upwind side),
//   q_n = u_n (q1 - r) + (L_n + R_n)/2 - cs d.
template <int DIR, bool FORCE = false>
__host__ __device__ __forceinline__ void riemann(const double (&L)[5], const double (&R)[5], const FaceRef& fr,
                                        double (&F)[5], double& un_out, bool up_forced = false) {
  AWFL_NO_CONTRACT
  constexpr int NM = 1 + DIR;
  constexpr int T1 = DIR == 0 ? 2 : 1;
  constexpr int T2 = DIR == 2 ? 2 : 3;
  const FaceAvg m = face_averages<DIR>(L, R);
  const double pw = pow_gamma_near(m.r * m.t, fm(m.r, m.t, -fr.rt.b) * fr.rt.rb, fr.rt.h, fr.rt.l);
  double cs, r2c;
  sqrt_halfrsqrt((GAMMA * C0) * pw * m.ir, cs, r2c);
  const bool up = FORCE ? up_forced : m.un > 0;
  const double u0 = up ? L[0] : R[0], u1 = up ? L[T1] : R[T1], u2 = up ? L[T2] : R[T2];
  const double D = fm(m.un, R[0] - L[0], L[NM] - R[NM]) * r2c;
  const double d = (R[4] - L[4]) * m.hit;
  const double v = D + (up ? d : -d);
  const double q1 = u0 + v;
  const double qn = fm(-cs, d, fm(m.un, q1 - m.r, 0.5 * (L[NM] + R[NM])));
  const double q5 = fm(m.t, D, 0.5 * (L[4] + R[4]));
  const double un1 = qn * rcp(q1);
  F[0] = qn;
  F[NM] = fm(qn, un1, C0 * pow_gamma_near(q5, (q5 - fr.q5.b) * fr.q5.rb, fr.q5.h, fr.q5.l));
  F[T1] = un1 * fm(m.ut1, v, u1);
  F[T2] = un1 * fm(m.ut2, v, u2);
  F[4] = un1 * q5;
  un_out = m.un;
}

template <int DIR>
__host__ __device__ __forceinline__ void riemann(const double (&L)[5], const double (&R)[5], const FaceRef& fr,
                                        double (&F)[5]) {
  double un;
  riemann<DIR>(L, R, fr, F, un);
}

// riemann(L, L): both sides of a wall face (S:822-823) are the cell's edge
// state, whose differences vanish; the remaining statements, bit for bit
template <int DIR>
__host__ __device__ __forceinline__ void wall_flux(const double (&L)[5], const FaceRef& fr, double (&F)[5]) {
  AWFL_NO_CONTRACT
  constexpr int NM = 1 + DIR;
  constexpr int T1 = DIR == 0 ? 2 : 1;
  constexpr int T2 = DIR == 2 ? 2 : 3;
  const double un1 = L[NM] * rcp(L[0]);
  F[0] = L[NM];
  F[NM] = fm(L[NM], un1, C0 * pow_gamma_near(L[4], (L[4] - fr.q5.b) * fr.q5.rb, fr.q5.h, fr.q5.l));
  F[T1] = un1 * L[T1];
  F[T2] = un1 * L[T2];
  F[4] = un1 * L[4];
}

}  // namespace awfl
