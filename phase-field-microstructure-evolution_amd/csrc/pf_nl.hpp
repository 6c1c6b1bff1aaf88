// The pointwise part of the FP64 faithful step, loops 5-10
// (src/var_diff.f90:685-905), in the reference's operation order.
#pragma once
#include "pf_step_kernels.hpp"

namespace pf {

constexpr int kNlRows = 4;  // rows i per pass over j

// Energies and extrema of the points a thread has taken.
struct NlDiag {
  double ch = 0.0, eta = 0.0, cmax = 0.0, cmin = 1.0, pmin = 1.0, p3 = 0.0;
};

// One point: con, and the V order parameters at ph[i * st], which are read while the
// results are given to put: put(0, df_dc), put(i + 1, df_dphi_i).  mob = mob_c -
// D_mean.
//   gamma_ij of src/var_diff.f90:206-218 (the matrix pf_gamma builds) is sigma_1
//   between two distinct matrix grains, sigma_2 between a grain and the precipitate
//   field eta_var (index mat) and 0 on the diagonal: the two values are used
//   directly, and a row's factor (2 gamma) phi_i, the same product for every j, is
//   formed once.  Every sum keeps the reference's order over i and j.
//   The pair sums read ph once per kNlRows rows i rather than once per pair: the LDS
//   traffic of the O(var^2) loops is what bounds them.
template <bool DIAG, typename Put>
__device__ __forceinline__ void nl_point_faithful(const UPar& u, int V, double con, const double* ph, int st, Put put,
                                                  double& mob, NlDiag& d) {
  const int mat = V - 1;
  // loop 5
  double fe = 0.0;
  if (DIAG) {
    for (int i = 0; i < V; ++i) {
      const double fi = ph[i * st], fi2 = fi * fi;
      fe = (fe - 0.5 * fi2) + 0.25 * (fi2 * fi2);
      const double g1 = u.s1g * fi2, g2 = u.s2g * fi2;
#pragma unroll 4
      for (int j = i + 1; j < mat; ++j) {
        const double fj = ph[j * st];
        fe = fe + g1 * (fj * fj);
      }
      if (i < mat) {
        const double fj = ph[mat * st];
        fe = fe + g2 * (fj * fj);
      }
    }
  }
  // loop 6
  double num = 0.0, den = 0.0;
#pragma unroll 4
  for (int i = 0; i < V; ++i) {
    const double f2 = ph[i * st] * ph[i * st], f4 = f2 * f2;
    if (i < mat) num = num + f4;
    den = den + f4;
  }
  const double hm = num / den, hp = 1.0 - hm;
  const double dm = con - u.cm, dp = con - u.cp;
  const double fch = (hm * u.am) * (dm * dm) + (hp * u.ap) * (dp * dp);
  put(0, ((2.0 * hm) * u.am) * dm + ((2.0 * hp) * u.ap) * dp);
  // loops 7-9
  const double fm = u.am * (dm * dm), fp = u.ap * (dp * dp);
  const double fv = ph[mat * st], fv2 = fv * fv, fv4 = fv2 * fv2;
  const double t2v = (4.0 * (fv2 * fv)) * (den - fv4);
  const double den2 = den * den;
  double ps = 0.0;
  for (int i0 = 0; i0 < mat; i0 += kNlRows) {
    double fi[kNlRows], ci[kNlRows], term2[kNlRows];
#pragma unroll
    for (int r = 0; r < kNlRows; ++r) {
      fi[r] = (i0 + r < mat) ? ph[(i0 + r) * st] : 0.0;
      ci[r] = (2.0 * u.s1g) * fi[r];
      term2[r] = 0.0;
    }
    auto add = [&](int j) {
      const double fj = ph[j * st], fj2 = fj * fj;
#pragma unroll
      for (int r = 0; r < kNlRows; ++r) term2[r] = term2[r] + ci[r] * fj2;
    };
#pragma unroll 4
    for (int j = 0; j < i0; ++j) add(j);
#pragma unroll
    for (int q = 0; q < kNlRows; ++q) {  // the rows' own block: no term j = i
      const double fj2 = fi[q] * fi[q];
#pragma unroll
      for (int r = 0; r < kNlRows; ++r)
        if (r != q) term2[r] = term2[r] + ci[r] * fj2;
    }
#pragma unroll 4
    for (int j = i0 + kNlRows; j < mat; ++j) add(j);
#pragma unroll
    for (int r = 0; r < kNlRows; ++r) {
      if (i0 + r >= mat) continue;
      const double f = fi[r];
      const double term1 = (f * f) * f - f;
      const double t2 = term2[r] + ((2.0 * u.s2g) * f) * fv2;
      const double term4 = (((4.0 * ((f * f) * f)) * fv4) * (fm - fp)) / den2;
      put(i0 + r + 1, (term1 + t2) + term4);
      ps = ps + f * f;
    }
  }
  {
    const double term1 = (fv * fv) * fv - fv, c2 = (2.0 * u.s2g) * fv;
    double t2 = 0.0;
#pragma unroll 4
    for (int j = 0; j < mat; ++j) {
      const double fj = ph[j * st];
      t2 = t2 + c2 * (fj * fj);
    }
    const double term4 = (t2v * (fp - fm)) / den2;
    put(V, (term1 + t2) + term4);
    ps = ps + fv * fv;
  }
  // loop 10: mob_c = D_bulk(var) + 2(1 - sum phi^2) D_gb, D_bulk(var) = D_L = D_mean;
  // loop 12 multiplies by mob_c - D_mean
  mob = (u.D + ((2.0 * (1.0 - ps)) * u.Dgb)) - u.D;
  if (DIAG) {
    d.ch += fch;
    d.eta += fe;
    if (fv > d.p3) d.p3 = fv;
    if (con <= d.cmin) d.cmin = con;
    if (con > d.cmax) d.cmax = con;
    if (ps < d.pmin) d.pmin = ps;
  }
}

// The same with the order parameters in registers, V <= kNlRegs: f holds the V - 1
// matrix grains, 0 from there on (terms of 0 that leave the sums as they are, and are
// skipped four at a time), fv the precipitate's.  Nothing is read after a result is
// given, so put may overwrite the point's values.
//   What is fused into a multiply-add is written out and nothing else is: left to the
//   compiler, the choice for products that the energies use too differed between the
//   two values of DIAG, and with it the last bits of the state between runs that report
//   other steps.
constexpr int kNlRegs = 16;
template <bool DIAG, typename Put>
__device__ __forceinline__ void nl_point_regs(const UPar& u, int V, double con, const double (&f)[kNlRegs], double fv,
                                              Put put, double& mob, double& ch, double& eta, double& cmax,
                                              double& cmin, double& pmin, double& p3) {
#pragma clang fp contract(off)
  const int mat = V - 1;
  const double fv2 = fv * fv, fv4 = fv2 * fv2;
  // loop 5
  double fe = 0.0;
  if (DIAG) {
#pragma unroll
    for (int i = 0; i < kNlRegs - 1; ++i) {
      if (i >= mat) break;
      const double fi2 = f[i] * f[i];
      fe = fma(0.25, fi2 * fi2, fma(-0.5, fi2, fe));
      const double g1 = u.s1g * fi2, g2 = u.s2g * fi2;
#pragma unroll
      for (int j0 = 0; j0 < kNlRegs; j0 += kNlRows) {
        if (j0 + kNlRows - 1 <= i || j0 >= mat) continue;
#pragma unroll
        for (int j = j0; j < j0 + kNlRows; ++j)
          if (j > i) fe = fma(g1, f[j] * f[j], fe);
      }
      fe = fma(g2, fv2, fe);
    }
    fe = fma(0.25, fv4, fma(-0.5, fv2, fe));
  }
  // loop 6
  double num = 0.0;
#pragma unroll
  for (int i = 0; i < kNlRegs; ++i) {
    const double f2 = f[i] * f[i];
    num = fma(f2, f2, num);
  }
  const double den = num + fv4;
  const double hm = num / den, hp = 1.0 - hm;
  const double dm = con - u.cm, dp = con - u.cp;
  const double fch = fma(hm * u.am, dm * dm, (hp * u.ap) * (dp * dp));
  put(0, fma((2.0 * hm) * u.am, dm, ((2.0 * hp) * u.ap) * dp));
  // loops 7-9
  const double fm = u.am * (dm * dm), fp = u.ap * (dp * dp);
  const double t2v = (4.0 * (fv2 * fv)) * (den - fv4);
  const double den2 = den * den;
  double ps = 0.0;
#pragma unroll
  for (int i0 = 0; i0 < kNlRegs; i0 += kNlRows) {
    if (i0 >= mat) continue;
#pragma unroll
    for (int i = i0; i < i0 + kNlRows; ++i) {
      if (i >= mat) break;
      const double fi = f[i], ci = (2.0 * u.s1g) * fi;
      double t2 = 0.0;
#pragma unroll
      for (int j0 = 0; j0 < kNlRegs; j0 += kNlRows) {
        if (j0 >= mat) continue;
#pragma unroll
        for (int j = j0; j < j0 + kNlRows; ++j)
          if (j != i) t2 = fma(ci, f[j] * f[j], t2);
      }
      const double term1 = fma(fi * fi, fi, -fi);
      t2 = fma((2.0 * u.s2g) * fi, fv2, t2);
      const double term4 = (((4.0 * ((fi * fi) * fi)) * fv4) * (fm - fp)) / den2;
      put(i + 1, (term1 + t2) + term4);
      ps = fma(fi, fi, ps);
    }
  }
  {
    const double term1 = fma(fv2, fv, -fv), c2 = (2.0 * u.s2g) * fv;
    double t2 = 0.0;
#pragma unroll
    for (int j = 0; j < kNlRegs; ++j) t2 = fma(c2, f[j] * f[j], t2);
    const double term4 = (t2v * (fp - fm)) / den2;
    put(V, (term1 + t2) + term4);
    ps = fma(fv, fv, ps);
  }
  // loop 10
  mob = fma(2.0 * (1.0 - ps), u.Dgb, u.D) - u.D;
  if (DIAG) {
    ch += fch;
    eta += fe;
    if (fv > p3) p3 = fv;
    if (con <= cmin) cmin = con;
    if (con > cmax) cmax = con;
    if (ps < pmin) pmin = ps;
  }
}

}  // namespace pf
