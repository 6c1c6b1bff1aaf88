// Definition of the x-line dispatch of pf_launch.hpp, for the files that
// instantiate it.
#pragma once
#include <algorithm>
#include <string>

#include "pf_launch.hpp"

namespace pf {

// Lines per x-line block: the smallest of 1, 2, 4, 8 that gives the block's
// transforms at least two waves of work (F*LINES*T >= 128 threads) and fills the
// lanes of a wave that moves rows (xline_rows_at_once: 96 x 96 lines of 64 points x
// 17 fields, 4 lines a block 25 us, 2 lines 34 us; of 128 points, 2 lines 46 us, 1
// line 58 us).  Small blocks keep several of them resident per CU, which is what
// hides the latency of each block's staging and barriers: at 256^3 x 17 fields one
// line per block (3 waves, 20 KB of LDS) runs 1.2x faster than two.
constexpr int kXlineMinThreads = 128;
inline int xline_lines(long F, int M, int cbytes) {
  int want = xline_rows_at_once(M, 8);
  while (want < 8 && F * want * xline_T(M, cbytes) < kXlineMinThreads) want *= 2;
  return want;
}

// LDS one x-line block may take (gfx950: 160 KiB per workgroup); above 64 KiB
// the kernel is opted in with hipFuncAttributeMaxDynamicSharedMemorySize.
constexpr size_t kXlineMaxLds = 160 * 1024;

template <typename R, int NX> size_t xline_lds(long jobs) {
  return sizeof(c2<R>) * ((size_t)jobs * xline_row_pitch(NX / 2, sizeof(c2<R>)) + NX);
}
// What is accepted: at most one block's threads with the default plan (whose
// thread count bounds the fields: 512-point lines, 64 in FP32 and, by LDS, 37 in
// FP64), and the rows in LDS (with 128 bytes to spare).
template <typename R, int NX> bool xline_fits(const Geo& g, long F, int lines) {
  const long jobs = F * lines;
  const long threads = std::max<long>(64, (jobs * plan_T(NX / 2) + 63) / 64 * 64);
  return g.plane % lines == 0 && threads <= kXlineMaxThreadsN<R, NX> &&
         xline_lds<R, NX>(jobs) + 16 * sizeof(double) <= kXlineMaxLds;
}

template <typename R, int NX, int LINES, bool XONLY, bool BATCH, bool KEEP, bool ROUNDS, bool FAITH = false>
int xline_one(const StepCall& c, c2<R>* wm, c2<R>* wn, R* mobd, double* part, long ngroups, long waves, bool diag,
              bool mob, const Member<R>* mt, long* nblocks, hipStream_t s) {
  const Geo& g = c.g;
  // with diagnostics every block leaves partials to reduce; 512-point lines set up
  // tables and register twiddles per block (512 x 128 x 128 x 37: 809 us with one
  // group a block, 783 us with two)
  const long cap = (!XONLY && c.tune.xline_grid > 0) ? c.tune.xline_grid
                   : (diag || NX >= 512)             ? kMaxGrid
                                                     : kXlineGroupCap;
  const long grid = xline_grid(ngroups, cap);
  const size_t shb = xline_lds<R, NX>((long)(XONLY ? 1 : g.F) * LINES);
  const c2<R>* tw = twiddle_table<R>(NX);
  if (!tw) return fail(PF_EHIP, "twiddle table set-up failed");
  auto kernel = &k_xline<R, NX, LINES, XONLY, BATCH, KEEP, ROUNDS, FAITH>;
  if (shb > 65536 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)shb) != hipSuccess)
    return fail(PF_EHIP, "x-line kernel: " + std::to_string(shb) + " bytes of LDS refused");
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3((unsigned)(64 * waves)), shb, s, g, c.u, wm, wn, mobd, tw,
                     part, ngroups, (int)diag, (int)mob, mt);
  if (nblocks) *nblocks = grid;
  return 0;
}

template <typename R, int NX, int LINES, bool XONLY, bool BATCH>
int xline_lines_of(const StepCall& c, c2<R>* wm, c2<R>* wn, R* mobd, double* part, long nmem, bool diag, bool mob,
                   const Member<R>* mt, long* nblocks, hipStream_t s) {
  const Geo& g = c.g;
  const long F = XONLY ? 1 : g.F, jobs = F * LINES, ngroups = nmem * (g.plane / LINES);
  constexpr int JW = xline_wave_jobs(NX / 2, sizeof(c2<R>));
  const long waves = (jobs + JW - 1) / JW, most = kXlineMaxThreadsN<R, NX> / 64;
  if (waves > most) {  // blocks of fewer lines, and in the end several rounds of the block's waves
    if constexpr (LINES > 1)
      return xline_lines_of<R, NX, LINES / 2, XONLY, BATCH>(c, wm, wn, mobd, part, nmem, diag, mob, mt, nblocks, s);
    else if constexpr (!XONLY)
      return xline_one<R, NX, 1, false, BATCH, false, true>(c, wm, wn, mobd, part, ngroups, most, diag, mob, mt,
                                                            nblocks, s);
  }
  // cache policy: W of every member, or the chain's one field beside the handle's
  if (bank_stays(sizeof(R) * (unsigned long)g.P * g.F * nmem))
    return xline_one<R, NX, LINES, XONLY, BATCH, true, false>(c, wm, wn, mobd, part, ngroups, waves, diag, mob, mt,
                                                              nblocks, s);
  return xline_one<R, NX, LINES, XONLY, BATCH, false, false>(c, wm, wn, mobd, part, ngroups, waves, diag, mob, mt,
                                                             nblocks, s);
}

template <typename R, bool XONLY, bool BATCH>
int xline_size(const StepCall& c, c2<R>* wm, c2<R>* wn, R* mobd, double* part, long nmem, bool diag, bool mob,
               const Member<R>* mt, long* nblocks, hipStream_t s) {
  const Geo& g = c.g;
  const long F = XONLY ? 1 : g.F;
  switch (g.nx) {
#define PF_TRY(N, L)             \
  if (xline_fits<R, N>(g, F, L)) \
    return xline_lines_of<R, N, L, XONLY, BATCH>(c, wm, wn, mobd, part, nmem, diag, mob, mt, nblocks, s);
#define PF_CASE(N)                                                                                           \
  case N: {                                                                                                  \
    const int tl = XONLY ? 0 : c.tune.xline_lines, want = tl > 0 ? tl : xline_lines(F, N / 2, sizeof(c2<R>)); \
    if (want == 8) { PF_TRY(N, 8) }                                                                          \
    if (want == 4 || (tl == 0 && want > 4)) { PF_TRY(N, 4) }                                                 \
    if (want == 2 || (tl == 0 && want > 2)) { PF_TRY(N, 2) }                                                 \
    if (want == 1 || tl == 0) { PF_TRY(N, 1) }                                                               \
    return fail(PF_ENOTIMPL, "x-line kernel: " + std::to_string(F) + " fields of length " #N " in " +        \
                                 std::to_string(want) + "-line blocks exceed one block's threads or LDS");   \
  }
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
#undef PF_TRY
    default: return fail(PF_EINVAL, "unsupported nx");
  }
}

template <typename R>
int xline(bool xonly, const StepCall& c, c2<R>* wm, c2<R>* wn, R* mobd, double* part, long* nblocks, bool diag,
          bool mob, hipStream_t s) {
  return xonly ? xline_size<R, true, false>(c, wm, wn, mobd, part, 1, diag, mob, nullptr, nblocks, s)
               : xline_size<R, false, false>(c, wm, wn, mobd, part, 1, diag, mob, nullptr, nblocks, s);
}

// The faithful step's x pass: a thread per point, one round.
template <int NX, int LINES>
int xline_faithful_lines(const StepCall& c, bool real, Bank<double> U, double* mobd, double* part, long* nblocks,
                         bool diag, hipStream_t s) {
  const Geo& g = c.g;
  constexpr int JW = xline_wave_jobs(NX / 2, sizeof(double2));
  const long jobs = (long)g.F * LINES, ngroups = g.plane / LINES;
  const long waves = std::max<long>((jobs + JW - 1) / JW, (LINES * NX + 63) / 64);
  // the state and derivative banks together
  if (bank_stays(2ul * g.F * g.P * sizeof(double)))
    return xline_one<double, NX, LINES, false, false, true, false, true>(c, U.main, U.nyq, mobd, part, ngroups, waves,
                                                                         diag, real, nullptr, nblocks, s);
  return xline_one<double, NX, LINES, false, false, false, false, true>(c, U.main, U.nyq, mobd, part, ngroups, waves,
                                                                        diag, real, nullptr, nblocks, s);
}
template <int NX>
int xline_faithful_of(const StepCall& c, bool real, Bank<double> U, double* mobd, double* part, long* nblocks,
                      bool diag, hipStream_t s) {
  const Geo& g = c.g;
  constexpr int JW = xline_wave_jobs(NX / 2, sizeof(double2)), threads = 512;
  const int want = xline_lines(g.F, NX / 2, sizeof(double2));
#define PF_TRY(L)                                                                              \
  if constexpr (L * NX <= threads)                                                             \
    if (want >= L && xline_fits<double, NX>(g, g.F, L) && (long)g.F * L <= JW * (threads / 64)) \
      return xline_faithful_lines<NX, L>(c, real, U, mobd, part, nblocks, diag, s);
  PF_TRY(8) PF_TRY(4) PF_TRY(2) PF_TRY(1)
#undef PF_TRY
  return fail(PF_ENOTIMPL, "faithful x line: fields exceed one block");
}

template <typename R> bool xline_accepts(const Geo& g, int lines) {
  switch (g.nx) {
#define PF_CASE(N) \
  case N:          \
    return lines ? xline_fits<R, N>(g, g.F, lines) : xline_fits<R, N>(g, g.F, 1);
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    default: return false;
  }
}

}  // namespace pf
