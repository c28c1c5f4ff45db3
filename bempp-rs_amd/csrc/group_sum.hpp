// group_sum.hpp -- the point-pair sums of one regular cell pair with the symmetric triangle rules
// taken as groups of three points (included by kernels.hpp).
//
// Every rule of triangle_rule is the centroid (or not) and groups of three points: an S21 orbit,
// or one of the two cyclic halves of an S111 orbit. Point k = 0, 1, 2 of a group has barycentric
// coordinate g + p at vertex k, g + s at vertex k + 1 and g at k + 2 (s = 0 for S21), so its
// offset from the centroid is p d_k + s d_{k+1}, d the cell's vertex offsets (d_0 + d_1 + d_2 = 0).
// With X = x_p - c the test point relative to the trial cell's centroid,
//   r^2 = |X|^2 + |o_q|^2 - 2 X.o_q = base + G_q - 2 p U_k - 2 s U_{k+1},  U_k = X.d_k,
// two instructions per point pair for S21 groups and three for the others instead of six, the
// trial cell being 6 values and its G_q; sums over the basis functions split the same way,
//   sum_q w K_q psi_b(q) = sum_groups (w p) K_b + (w s) K_{b-1} + (w g) (K_0 + K_1 + K_2).
#pragma once
#include <type_traits>

namespace bempp_amd {
namespace dev {

// Bound by FP64 VALU issue (88 to 96 % busy); a point pair of the 6-point rule on P1 costs 14.5 (Laplace
// double layer) to 30 (Helmholtz) instructions with its share of everything per test point and cell
// pair, against 22 and 43 with point coordinates, trial points in SGPRs (which spilled) and
// test points re-read per trial cell (which kept the vector L1 busy). Whole assemblies, near pairs included:
// Helmholtz hypersingular P1, 20480 cells, 6 points: 19.4 -> 11.8 ms; Laplace double layer P1, 19110
// cells: 12.0 -> 8.6 ms; Laplace single layer P1, 5120 cells, 16 points: 3.12 -> 1.64 ms;
// Helmholtz single layer P0, 5120 cells, 37 points: 17.7 -> 16.1 ms. Loops over a run-time number
// of groups two at a time measured the same.

// Fields of a group's record in the device table (RegularArgs::groups, kGroupStride doubles).
// The basis weights are those of the pair of spaces: a P0 side has wp = ws = 0, wg = w.
constexpr int kGroupStride = 12;
constexpr int kGrpP = 0, kGrpS = 1, kGrpM2P = 2, kGrpM2S = 3, kGrpW = 4, kGrpPP = 5;
constexpr int kGrpTest = 6;   // wp, ws, wg of the test side
constexpr int kGrpTrial = 9;  // of the trial side

// S21 and cyclic groups of the rules compiled with their point count; Q = 0 takes the counts
// from the arguments (rules of 16 and 37 points: 3 + 2 and 4 + 8 groups and the centroid).
template <int Q>
constexpr int kGroups21 = Q == 3 ? 1 : (Q == 6 || Q == 7) ? 2 : 0;
template <int Q>
constexpr bool kHasCentroid = Q == 0 || Q == 1 || Q == 7;

// Kernel value of a point pair in scaled form: from h = (kappa / 2)^2 r^2 (centred Helmholtz,
// kappa = |k|) or h = r^2, one Newton step y (3 - h y^2) of y = rsq(h) without its factor 1/2
// gives rz = 4 / (kappa r) or 2 / r, and h rz = kappa r or 2 r: the phase costs one FMA. The
// caller multiplies sums by group_factor and, for k < 0, conjugates. dn (adjoint double layer):
// as kernel_scalar_r2; the double layer's (x - y).n_y is the same for every y of the flat trial
// cell and is left to the caller.
template <int OP, bool HELM, int TIER>
__device__ __forceinline__ cplx group_kernel(double h, double dn, double kR, double khalf) {
  const double y = __builtin_amdgcn_rsq(h);
  const double rz = y * fma(-(h * y), y, 3.0);
  if constexpr (!HELM) {
    if constexpr (OP == 0 || OP == 3) return {rz, 0.0};
    else if constexpr (OP == 1) return {rz * (rz * rz), 0.0};
    else return {(dn * rz) * (rz * rz), 0.0};
  } else {
    double s, c, kr;
    if constexpr (TIER > 0) {
      if constexpr (OP == 0 || OP == 3) {
        sincos_small<TIER>(fma(h, rz, -kR), &s, &c);
        kr = 0.0;
      } else {
        kr = h * rz;
        sincos_small<TIER>(kr - kR, &s, &c);
      }
    } else {
      kr = (h * rz) * khalf;
      sincos_cw(kr, &s, &c);
    }
    if constexpr (OP == 0 || OP == 3) {
      return {c * rz, s * rz};
    } else {
      const double f = (OP == 1 ? rz : dn * rz) * (rz * rz);
      return {fma(kr, s, c) * f, fma(-kr, c, s) * f};
    }
  }
}

// Whether lengths can be scaled by |k| for cells of this radius (host): (kappa / 2)^2 r^2 must not
// underflow, nor (4 / (kappa r))^3 and its factor (kappa / 4)^3 leave the range, with room for point pairs
// much nearer than the radius. Other wavenumbers, k = 0 among them, take phase tier 0, which is unscaled.
inline bool scalable(double k, double radius) {
  const double kappa = k < 0.0 ? -k : k;
  return kappa >= 1e-80 && kappa * radius >= 1e-80;
}

// Whether a cell pair is too near for r^2 by terms (R2 the squared centroid distance, radii the sum of
// the two cells' radii). From 1.25 radius sums on a point pair has at least r = (1.25 - t) radii, t the
// rules' largest point radius (0.73 compiled, 0.98 others), and |X| + |o_q| <= (1.25 + t) radii: the terms'
// roundings count at most 15 (65) times in r^2, at the one extreme pair. Neighbours that do not touch are
// 1.32 radius sums apart in a triangulation of equilateral cells (1.41: squares) and nearer where it is
// graded or stretched or sheets of it lie close; by terms r^2 is wrong by (size / r)^2 roundings there,
// and not positive at last.
constexpr double kGroupNear = 1.25 * 1.25;
__device__ __forceinline__ bool group_near(double R2, double radii) { return R2 < kGroupNear * (radii * radii); }

template <int OP, bool HELM, int TIER>
__device__ __forceinline__ double group_factor(double kappa) {
  const double f = HELM && TIER > 0 ? 0.25 * kappa : 0.5;
  return OP == 0 || OP == 3 ? f : f * f * f;
}

__device__ __forceinline__ void add_scaled(cplx& a, cplx v, double f) {
  a.re = fma(v.re, f, a.re);
  a.im = fma(v.im, f, a.im);
}

// One test point X (relative to the trial centroid) against every trial point: T_b(p) (P1) or
// the weighted sum in T[0]. dn: -(x_p - c).n_x, with nk[k] = d_k.n_x (adjoint double layer). d: d_0, d_1; g: |d_k|^2 (compiled rules); gq: G of the cell's grouped
// points (Q = 0); sc: (kappa / 2)^2 or 1.
template <int Q, int OP, bool HELM, int TIER, bool P1, typename Args, typename GQ>
__device__ __forceinline__ void group_trial_sum(Args& A, const double (&X)[3], double dn, const double (&nk)[3],
                                                const double (&d)[2][3], const double (&g)[3], GQ gq, double sc,
                                                double kR, double khalf, cplx (&T)[P1 ? 3 : 1]) {
  constexpr bool SC = HELM && TIER > 0;
  const double Xs[3] = {SC ? X[0] * sc : X[0], SC ? X[1] * sc : X[1], SC ? X[2] * sc : X[2]};
  const double base = X[0] * Xs[0] + X[1] * Xs[1] + X[2] * Xs[2];
  double U[3];
  U[0] = Xs[0] * d[0][0] + Xs[1] * d[0][1] + Xs[2] * d[0][2];
  U[1] = Xs[0] * d[1][0] + Xs[1] * d[1][1] + Xs[2] * d[1][2];
  U[2] = -(U[0] + U[1]);
  const auto tab = constant_view(A.groups);
  cplx S = {0.0, 0.0};  // P1: the sum of (w g) K
#pragma unroll
  for (int b = 0; b < (P1 ? 3 : 1); ++b) T[b] = {0.0, 0.0};
  if constexpr (kHasCentroid<Q>) {
    if (Q != 0 || A.wc != 0.0) {
      const cplx kv = group_kernel<OP, HELM, TIER>(base, dn, kR, khalf);
      if constexpr (P1) add_scaled(S, kv, A.wc_trial);
      else add_scaled(T[0], kv, A.wc);
    }
  }
  auto group = [&](const auto* r, auto cyclic, const double (&gk)[3]) {
    const double mp = r[kGrpM2P], ms = r[kGrpM2S];
    cplx acc = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      double h = fma(mp, U[k], gk[k]);
      double dq = dn;
      if constexpr (decltype(cyclic)::value) h = fma(ms, U[(k + 1) % 3], h);
      if constexpr (OP == 2) {
        dq = fma(r[kGrpP], nk[k], dq);
        if constexpr (decltype(cyclic)::value) dq = fma(r[kGrpS], nk[(k + 1) % 3], dq);
      }
      const cplx kv = group_kernel<OP, HELM, TIER>(h, dq, kR, khalf);
      if constexpr (P1) {
        add_scaled(T[k], kv, r[kGrpTrial]);
        if constexpr (decltype(cyclic)::value) add_scaled(T[(k + 1) % 3], kv, r[kGrpTrial + 1]);
        add_scaled(S, kv, r[kGrpTrial + 2]);
      } else {
        acc.re += kv.re;
        acc.im += kv.im;
      }
    }
    if constexpr (!P1) add_scaled(T[0], acc, r[kGrpW]);
  };
  if constexpr (Q != 0) {
#pragma unroll
    for (int m = 0; m < kGroups21<Q>; ++m) {
      const auto r = tab + m * kGroupStride;
      const double pp = SC ? sc * r[kGrpPP] : r[kGrpPP];  // invariant over test points
      const double gk[3] = {fma(pp, g[0], base), fma(pp, g[1], base), fma(pp, g[2], base)};
      group(r, std::false_type{}, gk);
    }
  } else {
    int m = 0;
#pragma unroll 1
    for (; m < A.n21; ++m) {
      const auto q = gq + 3 * m;
      const double gk[3] = {SC ? fma(sc, q[0], base) : base + q[0], SC ? fma(sc, q[1], base) : base + q[1],
                            SC ? fma(sc, q[2], base) : base + q[2]};
      group(tab + m * kGroupStride, std::false_type{}, gk);
    }
#pragma unroll 1
    for (; m < A.ngroups; ++m) {
      const auto q = gq + 3 * m;
      const double gk[3] = {SC ? fma(sc, q[0], base) : base + q[0], SC ? fma(sc, q[1], base) : base + q[1],
                            SC ? fma(sc, q[2], base) : base + q[2]};
      group(tab + m * kGroupStride, std::true_type{}, gk);
    }
  }
  if constexpr (P1)
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      T[b].re += S.re;
      T[b].im += S.im;
    }
}

// The sums of one cell pair without Jacobians, group_factor, conjugation, e^{ikR} and 1/(4 pi):
// P1: M_ab = sum_pq w_p w_q phi_a(p) psi_b(q) K_pq; otherwise M[0][0] = sum_pq w_p w_q K_pq.
// td: the test cell's vertex offsets d'_0, d'_1; D: test centroid minus trial centroid.
template <int Q, int OP, bool HELM, int TIER, bool P1, typename Args, typename GQ>
__device__ __forceinline__ void group_pair_sum(Args& A, const double (&td)[2][3], const double (&D)[3],
                                               const double (&nx)[3], const double (&ny)[3], const double (&d)[2][3],
                                               const double (&g)[3], GQ gq, double kappa, double kR,
                                               cplx (&M)[P1 ? 3 : 1][P1 ? 3 : 1]) {
  constexpr int NB = P1 ? 3 : 1;
  const double khalf = 0.5 * kappa;
  const double sc = HELM && TIER > 0 ? khalf * khalf : 1.0;
  double Dn = 0.0, nk[3] = {0.0, 0.0, 0.0};
  if constexpr (OP == 2) {
    Dn = -(D[0] * nx[0] + D[1] * nx[1] + D[2] * nx[2]);
    nk[0] = d[0][0] * nx[0] + d[0][1] * nx[1] + d[0][2] * nx[2];
    nk[1] = d[1][0] * nx[0] + d[1][1] * nx[1] + d[1][2] * nx[2];
    nk[2] = -(nk[0] + nk[1]);
  }
  const double dt[3][3] = {{td[0][0], td[0][1], td[0][2]},
                           {td[1][0], td[1][1], td[1][2]},
                           {-(td[0][0] + td[1][0]), -(td[0][1] + td[1][1]), -(td[0][2] + td[1][2])}};
  cplx C[NB];  // P1: the part of M common to its rows
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    C[a] = {0.0, 0.0};
#pragma unroll
    for (int b = 0; b < NB; ++b) M[a][b] = {0.0, 0.0};
  }
  // returns the factor of the test point's weight: (x_p - y).n_y for the double layer, else 1
  auto point = [&](const double (&X)[3], cplx (&T)[NB]) {
    group_trial_sum<Q, OP, HELM, TIER, P1>(A, X, Dn, nk, d, g, gq, sc, kR, khalf, T);
    return OP == 1 ? X[0] * ny[0] + X[1] * ny[1] + X[2] * ny[2] : 1.0;
  };
  if constexpr (kHasCentroid<Q>) {
    if (Q != 0 || A.wc != 0.0) {
      cplx T[NB];
      const double dn = point(D, T);
      const double w = P1 ? A.wc_test : A.wc;
#pragma unroll
      for (int b = 0; b < NB; ++b) add_scaled(C[b], T[b], OP == 1 ? w * dn : w);
    }
  }
  const auto tab = constant_view(A.groups);
  auto group = [&](const auto* r, auto cyclic) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      constexpr bool CY = decltype(cyclic)::value;
      double X[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        X[c] = fma(r[kGrpP], dt[k][c], D[c]);
        if constexpr (CY) X[c] = fma(r[kGrpS], dt[(k + 1) % 3][c], X[c]);
      }
      cplx T[NB];
      const double dn = point(X, T);
      auto weight = [&](double w) { return OP == 1 ? w * dn : w; };
      if constexpr (P1) {
        const double wp = weight(r[kGrpTest]), ws = CY ? weight(r[kGrpTest + 1]) : 0.0, wg = weight(r[kGrpTest + 2]);
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          add_scaled(M[k][b], T[b], wp);
          if constexpr (CY) add_scaled(M[(k + 1) % 3][b], T[b], ws);
          add_scaled(C[b], T[b], wg);
        }
      } else {
        add_scaled(C[0], T[0], weight(r[kGrpW]));
      }
    }
  };
  const int n21 = Q != 0 ? kGroups21<Q> : A.n21;
#pragma unroll 1
  for (int m = 0; m < n21; ++m) group(tab + m * kGroupStride, std::false_type{});
  if constexpr (Q == 0)
#pragma unroll 1
    for (int m = A.n21; m < A.ngroups; ++m) group(tab + m * kGroupStride, std::true_type{});
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      M[a][b].re += C[b].re;
      M[a][b].im += C[b].im;
    }
}

// The sums of group_pair_sum (group_factor applied) of a pair of near cells, r^2 from the differences
// X - o_q = D + (x_p - c') - (y_q - c). The kernels note the near trial cells of each lane and take them
// after the far ones, each lane its own (d and ny per lane): Laplace single layer P1, 16-point rule, 5120
// cells, where 1.3 % of the trial cells of a wavefront have a near lane, takes 1.53 ms without near pairs
// by differences, 1.64 so, 1.93 with the whole wavefront's pairs by differences where one lane is near.
template <int OP, bool HELM, int TIER, bool P1, typename Args>
__device__ __forceinline__ void near_pair_sum(Args& A, const double (&td)[2][3], const double (&D)[3],
                                              const double (&nx)[3], const double (&ny)[3], const double (&d)[2][3],
                                              double kappa, double kR, cplx (&M)[P1 ? 3 : 1][P1 ? 3 : 1]) {
  constexpr int NB = P1 ? 3 : 1;
  const auto tab = constant_view(A.rule_tab);  // barycentric coordinates and weight of each point
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) M[a][b] = {0.0, 0.0};
#pragma unroll 1
  for (int p = 0; p < A.nq; ++p) {
    const double l0 = tab[4 * p] - tab[4 * p + 2], l1 = tab[4 * p + 1] - tab[4 * p + 2];
    double X[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) X[c] = fma(l0, td[0][c], fma(l1, td[1][c], D[c]));
    cplx T[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) T[b] = {0.0, 0.0};
#pragma unroll 2
    for (int q = 0; q < A.nq; ++q) {
      const double m0 = tab[4 * q + 2] - tab[4 * q], m1 = tab[4 * q + 2] - tab[4 * q + 1];
      double r[3];
#pragma unroll
      for (int c = 0; c < 3; ++c) r[c] = fma(m0, d[0][c], fma(m1, d[1][c], X[c]));
      const cplx kv = kernel_scalar<OP, HELM, TIER>(r[0], r[1], r[2], kappa, nx, ny, kR);
#pragma unroll
      for (int b = 0; b < NB; ++b)
        add_scaled(T[b], kv, tab[4 * q + 3] * (P1 && A.nbs == 3 ? tab[4 * q + b] : b == 0 ? 1.0 : 0.0));
    }
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      const double w = tab[4 * p + 3] * (P1 && A.nbt == 3 ? tab[4 * p + a] : a == 0 ? 1.0 : 0.0);
#pragma unroll
      for (int b = 0; b < NB; ++b) add_scaled(M[a][b], T[b], w);
    }
  }
}

}  // namespace dev
}  // namespace bempp_amd
