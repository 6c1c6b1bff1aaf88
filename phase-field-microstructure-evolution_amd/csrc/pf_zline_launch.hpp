// Definition of the z-line dispatch of pf_launch.hpp, for the files that
// instantiate it.
#pragma once
#include <algorithm>
#include <string>

#include "pf_launch.hpp"

namespace pf {

// Cache policy of a pass over banks of nfields fields (k_zline's KEEP).
template <typename R> int zline_keep(const Geo& g, long nfields) {
  const unsigned long wb = (unsigned long)nfields * g.P * sizeof(R);
  return !bank_stays(wb) ? 0 : bank_stays(2 * wb) ? 2 : 1;
}

template <typename R, int N, int ROLE, bool DC64, bool PARSEVAL, bool BATCH, int V, int KEEP>
int zline_one(const StepCall& c, Bank<R> S, Bank<R> W, Bank<R> X, Bank<R> Y, double* dc64, double* part, int f0, int nf,
              const Member<R>* mt, long* nblocks, hipStream_t s) {
  const Geo& g = c.g;
  constexpr int TX = col_tile(N, sizeof(c2<R>));
  const long tm = ((long)g.M * g.ny + TX - 1) / TX, tn = ((long)g.ny + TX - 1) / TX;
  const long cap = c.tune.zline_grid > 0 ? c.tune.zline_grid : kZlineMaxGrid;
  long grid = std::min<long>((tm + tn) * nf, cap);
  // whole XCD runs of main-block rows (xcd_runs): extra blocks find no tile
  const long rows = c.tune.zline_run_rows < 0 ? 1 : c.tune.zline_run_rows;
  const long runt = rows * (((long)g.M + TX - 1) / TX), run = 8 * runt;
  if (run > 0 && (grid + run - 1) / run * run <= cap) grid = (grid + run - 1) / run * run;
  const c2<R>* tw = twiddle_table<R>(N);
  if (!tw) return fail(PF_EHIP, "twiddle table set-up failed");
  hipLaunchKernelGGL((k_zline<R, N, ROLE, DC64, PARSEVAL, BATCH, V, KEEP>), dim3((unsigned)grid),
                     dim3(TX * plan_T(N, V)), 0, s, g, c.u, c.kt, S, W, X, Y, dc64, part, tw, f0, nf, tm, tn, runt,
                     mt);
  if (nblocks) *nblocks = grid;
  return 0;
}

// The plan variant of a tuned shape (FP32 ROLE_REG), else the default plan.
template <typename R, int N, int ROLE, bool DC64, bool PARSEVAL, bool BATCH, int KEEP>
int zline_plan(const StepCall& c, Bank<R> S, Bank<R> W, Bank<R> X, Bank<R> Y, double* dc64, double* part, int f0, int nf,
               const Member<R>* mt, long* nblocks, hipStream_t s) {
  if constexpr (sizeof(R) == 4 && ROLE == ROLE_REG && plan_alt(N, 1, 0) != 0) {
    if (c.tune.zline_plan == 1)
      return zline_one<R, N, ROLE, DC64, PARSEVAL, BATCH, 1, KEEP>(c, S, W, X, Y, dc64, part, f0, nf, mt, nblocks, s);
    if (c.tune.zline_plan == 2)
      return zline_one<R, N, ROLE, DC64, PARSEVAL, BATCH, 2, KEEP>(c, S, W, X, Y, dc64, part, f0, nf, mt, nblocks, s);
  }
  return zline_one<R, N, ROLE, DC64, PARSEVAL, BATCH, 0, KEEP>(c, S, W, X, Y, dc64, part, f0, nf, mt, nblocks, s);
}

template <typename R, int ROLE, bool DC64, bool PARSEVAL, bool BATCH>
int zline_size(const StepCall& c, Bank<R> S, Bank<R> W, Bank<R> X, Bank<R> Y, double* dc64, double* part, int f0, int nf,
               const Member<R>* mt, long* nblocks, hipStream_t s) {
  const int keep = zline_keep<R>(c.g, BATCH ? nf : c.g.F);
  switch (c.g.nz) {
#define PF_CASE(N)                                                                                                 \
  case N:                                                                                                          \
    return keep == 2   ? zline_plan<R, N, ROLE, DC64, PARSEVAL, BATCH, 2>(c, S, W, X, Y, dc64, part, f0, nf, mt,   \
                                                                           nblocks, s)                             \
           : keep == 1 ? zline_plan<R, N, ROLE, DC64, PARSEVAL, BATCH, 1>(c, S, W, X, Y, dc64, part, f0, nf, mt,   \
                                                                           nblocks, s)                             \
                       : zline_plan<R, N, ROLE, DC64, PARSEVAL, BATCH, 0>(c, S, W, X, Y, dc64, part, f0, nf, mt,   \
                                                                           nblocks, s);
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    default: return fail(PF_EINVAL, "unsupported nz");
  }
}

template <typename R>
int zline(int role, bool parseval, const StepCall& c, Bank<R> S, Bank<R> W, Bank<R> X, Bank<R> Y, double* dc64,
          double* part, int f0, int nf, long* nblocks, hipStream_t s) {
  constexpr bool DC = sizeof(R) == 4;
  if (role == ROLE_GHAT)
    return zline_size<R, ROLE_GHAT, false, false, false>(c, S, W, X, Y, dc64, part, f0, nf, nullptr, nblocks, s);
  if (role == ROLE_CMOB)
    return parseval
               ? zline_size<R, ROLE_CMOB, DC, true, false>(c, S, W, X, Y, dc64, part, f0, nf, nullptr, nblocks, s)
               : zline_size<R, ROLE_CMOB, DC, false, false>(c, S, W, X, Y, dc64, part, f0, nf, nullptr, nblocks, s);
  return parseval ? zline_size<R, ROLE_REG, DC, true, false>(c, S, W, X, Y, dc64, part, f0, nf, nullptr, nblocks, s)
                  : zline_size<R, ROLE_REG, DC, false, false>(c, S, W, X, Y, dc64, part, f0, nf, nullptr, nblocks, s);
}

}  // namespace pf
