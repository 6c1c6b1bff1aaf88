// Kernels of the FP64 faithful step: the reference's loops 5-14 in FP64 on the
// real-space state, with its operation order per point and per mode.
#include <algorithm>

#include "../../include/pf.h"
#include "pf_internal.hpp"
#include "pf_faithful.hpp"
#include "pf_nl.hpp"
#include "pf_passes.hpp"

namespace pf {

// ---------------------------------------------------------------------------
// Loops 5-10 (src/var_diff.f90:685-905), O(var^2) per point.
// Reads the real state bank (c, eta_i); writes df_dc and df_dphi_i (a bank in the
// same order) and mob_c - D_mean.
//   A point's order parameters sit in the thread's own LDS column.  The pair sums
//   read it once per kNlRows rows i rather than once per pair: the LDS traffic of
//   the O(var^2) loops bounded the kernel.  256^3 x 17: 1.87 -> 0.84 ms, with the
//   energies 2.49 -> 1.03 ms; 0.84 ms is 5.6 TB/s over the 4.7 GB it moves, the
//   rate of a plain stream.
// ---------------------------------------------------------------------------
template <bool DIAG>
__global__ void __launch_bounds__(kNlBlock)
k_nl_faithful(Geo g, UPar u, const double* __restrict__ st, double* __restrict__ dfd, double* __restrict__ mobd,
              double* __restrict__ part) {
  constexpr int NB = kNlBlock;
  extern __shared__ double sh[];  // var * NB values, then NB reduction scratch
  double* red = sh + (long)g.var * NB;
  const int V = g.var;
  double* const ph = sh + threadIdx.x;
  NlDiag d;
  // cache policy of the state and derivative banks together
  const bool keep = bank_stays(2ul * (unsigned)g.F * g.P * sizeof(double));
  auto put = [&](double x, double* p) {
    if (keep) *p = x;
    else __builtin_nontemporal_store(x, p);
  };
  for (long t = (long)blockIdx.x * NB + threadIdx.x; t < g.P; t += (long)gridDim.x * NB) {
    if (keep) {
#pragma unroll 8
      for (int i = 0; i < V; ++i) ph[i * NB] = st[(long)(i + 1) * g.P + t];
    } else {
#pragma unroll 8
      for (int i = 0; i < V; ++i) ph[i * NB] = __builtin_nontemporal_load(st + (long)(i + 1) * g.P + t);
    }
    const double con = st[t];
    double mob;
    nl_point_faithful<DIAG>(u, V, con, ph, NB, [&](int f, double x) { put(x, dfd + (long)f * g.P + t); }, mob, d);
    mobd[t] = mob;
  }
  if (DIAG) {
    const double s0 = block_sum<NB>(d.ch, red), s1 = block_sum<NB>(d.eta, red);
    const double e0 = block_ext<NB, true>(d.cmax, red), e1 = block_ext<NB, false>(d.cmin, red);
    const double e2 = block_ext<NB, false>(d.pmin, red), e3 = block_ext<NB, true>(d.p3, red);
    if (threadIdx.x == 0) {
      double* o = part + (long)blockIdx.x * 6;
      o[0] = s0; o[1] = s1; o[2] = e0; o[3] = e1; o[4] = e2; o[5] = e3;
    }
  }
}

// ---------------------------------------------------------------------------
// k_zfaithful: everything that happens to a z column in k-space, one pass:
//   FZ_ETA : forward z of phi_i and of df_dphi_i, loop 14, inverse z of the new
//            phi_i.  3 banks over HBM; as separate transforms and a pointwise pass
//            it was 9.  256^3 x 17: 4.0 -> 1.37 ms, 4.7 TB/s
//   FZ_GHAT: forward z of c and of df_dc, left in their banks for FZ_CMOB; loop
//            11's g^ = kf_sum f^ - kappa_c c^ k_cube, inverse z of it -> G
//   FZ_CMOB: forward z of G, loop 13, inverse z of the new c
// PARS (FZ_ETA, FZ_GHAT): also loops 1-4's f_int of the state whose spectrum the
// pass holds, sum 0.5 kappa |grad u|^2 over the points, as Parseval's sum
// 0.5 kappa P sum_k w |kf|^2 |u^|^2 with the Nyquist-zeroed kf (w = 2 for the
// modes whose conjugates are not stored): the inverse transforms of the 3(var+1)
// gradient fields, 7.2 ms of a reported step at 256^3 x 17, are not needed; the
// sums cost 0.05 ms.
// Wavenumbers and updates are evaluated in the reference's order
// (src/var_diff.f90:932-935, 978-987, 1019-1027).
// A thread holds two columns' worth of values (2 x 64 VGPRs at 256 points): 2
// waves per SIMD, which the 64 KiB exchange tile allows too.  FZ_CMOB, one field of
// F, holds three and spills 15 VGPRs a lane at 128 points, 9 at 32 and 6 at 256.
// ---------------------------------------------------------------------------
__device__ __forceinline__ KCol<double> kcol_ref(const KTab& t, int kx, int ky) {
#pragma clang fp contract(off)
  const double ax = t.ax[kx], axp = t.axp[kx], ay = t.ay[ky], ayp = t.ayp[ky];
  const double x2 = ax * ax, y2 = ay * ay;
  KCol<double> c;
  c.s1 = axp + ayp;
  c.k2 = -x2 + -y2;
  c.k3 = -(axp * x2) + -(ayp * y2);
  c.k4 = (x2 * ax) * ax + (y2 * ay) * ay;
  c.kp2 = axp * axp + ayp * ayp;
  return c;
}
__device__ __forceinline__ KCoefR<double> kcoef_ref(const KCol<double>& c, int kz, int nz, double uz) {
#pragma clang fp contract(off)
  const double az = az_of(kz, nz, uz), azp = (2 * kz == nz) ? 0.0 : az;
  const double z2 = az * az;
  KCoefR<double> k;
  k.s1 = c.s1 + azp;
  k.k2 = c.k2 + -z2;
  k.k3 = c.k3 + -(azp * z2);
  k.k4 = c.k4 + (z2 * az) * az;
  k.kp2 = c.kp2 + azp * azp;
  return k;
}

template <int NZ, int ROLE, bool PARS, bool KEEP>
__global__ void __launch_bounds__(col_tile(NZ, sizeof(double2)) * plan_T(NZ)) __attribute__((amdgpu_waves_per_eu(2)))
k_zfaithful(Geo g, UPar u, KTab kt, Bank<double> U, Bank<double> D, Bank<double> G, double* __restrict__ part,
            const double2* __restrict__ tw, int f0, int nf, unsigned tm, unsigned tn, unsigned run_tiles) {
  using R = double;
  constexpr int TX = col_tile(NZ, sizeof(double2));
  constexpr int NI = kInSlots<NZ>, NO = kOutSlots<NZ>, E = plan_E(NZ);
  constexpr unsigned CB = sizeof(double2);
  constexpr int AUX = KEEP ? 0 : kBufNT;  // cache policy (bank_stays)
  static_assert(last_pass_in_place<NZ>(), "slot rows of the last pass are t + a per-slot constant");
  constexpr int SHN = (plan_np(NZ) > 1 || !rfft_io_same<NZ>()) ? NZ * TX : 1;
  __shared__ double2 sh[SHN * sizeof(double2) >= 16 * sizeof(double) ? SHN : 16 * sizeof(double) / sizeof(double2)];
  const unsigned tpf = tm + tn, total = (unsigned)nf * tpf;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const double ldt = u.L * u.dt, lkd = (u.L * u.kphi) * u.dt, Dk = (u.D * u.dt) * u.kc;
  double acc = 0.0;
  for (unsigned tile = (unsigned)xcd_runs(blockIdx.x, gridDim.x, run_tiles); tile < total; tile += gridDim.x) {
    const unsigned fi = tile / tpf, tt = tile - fi * tpf;
    const long f = f0 + (long)fi;
    const bool isn = tt >= tm;
    const unsigned Wd = isn ? (unsigned)g.ny : (unsigned)g.M * (unsigned)g.ny;
    const unsigned col0 = (isn ? tt - tm : tt) * TX;
    const bool act = col0 + c < Wd;
    const unsigned rowb = Wd * CB, nb = (unsigned)NZ * rowb;
    const long fo = (isn ? f * g.plane : f * g.hmain) + col0;
    const BufRes ru = buf_res((isn ? U.nyq : U.main) + fo, nb);
    const BufRes rd = buf_res((isn ? D.nyq : D.main) + fo, nb);
    const BufRes rg = buf_res((isn ? G.nyq : G.main) + col0, nb);  // one field
    const unsigned lw = ((unsigned)t * Wd + (unsigned)c) * CB;
    // 1. all loads of the tile: both transforms' inputs, or one's and c^, f^ at the output rows
    double2 a[E], b[E];
    double2 fh[ROLE == FZ_CMOB ? NO : 1];
#pragma unroll
    for (int s = 0; s < NI; ++s)
      if (act && rfft_in_valid<NZ>(t, s)) {
        const unsigned o = (unsigned)rfft_in_idx<NZ>(0, s) * rowb;
        if constexpr (ROLE == FZ_CMOB) {
          b[s] = buf_ld<R, AUX>(rg, lw, o);
        } else {
          b[s] = buf_ld<R, AUX>(rd, lw, o);
          a[s] = buf_ld<R, AUX>(ru, lw, o);
        }
      }
    if constexpr (ROLE == FZ_CMOB) {
#pragma unroll
      for (int s = 0; s < NO; ++s)
        if (act && rfft_out_valid<NZ>(t, s)) {
          const unsigned o = (unsigned)rfft_out_idx<NZ>(0, s) * rowb;
          a[s] = buf_ld<R, AUX>(ru, lw, o);
          fh[s] = buf_ld<R, AUX>(rd, lw, o);
        }
    }
    const int col = (int)col0 + c;
    const int kx = isn ? g.M : col % g.M, ky = act ? (isn ? col : col / g.M) : 0;
    const KCol<double> kc = kcol_ref(kt, kx, ky);
    int tz = t;  // opaque: the z wavenumbers are recomputed per tile, not hoisted into registers
    asm volatile("" : "+v"(tz));
    // 2. forward z, update in registers
    rfft<R, NZ, false, TX>(b, t, act, sh + c, tw);
    if constexpr (ROLE != FZ_CMOB) rfft<R, NZ, false, TX>(a, t, act, sh + c, tw);
    if (PARS) {
      double p1 = 0.0, p2 = 0.0;
#pragma unroll
      for (int s = 0; s < NO; ++s) {
        if (!(act && rfft_out_valid<NZ>(t, s))) continue;
        const int ez = rfft_out_idx<NZ>(tz, s);
        const double zp = (2 * ez == NZ) ? 0.0 : az_of(ez, NZ, kt.uz);
        const double m2 = a[s].x * a[s].x + a[s].y * a[s].y;
        p1 += m2;
        p2 += (zp * zp) * m2;
      }
      const double wgt = (kx == 0 || kx == g.M) ? 1.0 : 2.0;
      acc += (0.5 * (ROLE == FZ_GHAT ? u.kc : u.kphi)) * wgt * (kc.kp2 * p1 + p2);
    }
#pragma unroll
    for (int s = 0; s < NO; ++s) {
      if (!(act && rfft_out_valid<NZ>(t, s))) continue;
      const unsigned o = (unsigned)rfft_out_idx<NZ>(0, s) * rowb;
      const KCoefR<double> k = kcoef_ref(kc, rfft_out_idx<NZ>(tz, s), NZ, kt.uz);
      const double2 sa = a[s], sb = b[s];
      if constexpr (ROLE == FZ_ETA) {
        const double t22 = 1.0 - lkd * k.k2;
        a[s] = make_double2((sa.x - ldt * sb.x) / t22, (sa.y - ldt * sb.y) / t22);
      } else if constexpr (ROLE == FZ_GHAT) {
        buf_st<R, 0>(ru, lw, o, sa);  // c^
        buf_st<R, 0>(rd, lw, o, sb);  // f^
        const double kcr = u.kc * sa.x, kci = u.kc * sa.y;
        a[s] = make_double2(-(k.s1 * sb.y) - (-(kci * k.k3)), (k.s1 * sb.x) - (kcr * k.k3));
      } else {
        const double2 fs = fh[s];
        const double t11r = -((sb.y * u.dt) * k.s1), t11i = (sb.x * u.dt) * k.s1;
        const double t22 = 1.0 + Dk * k.k4;
        const double r33 = (u.D * k.k2) * u.dt;
        const double nr = (sa.x + t11r) + r33 * fs.x, ni = (sa.y + t11i) + r33 * fs.y;
        a[s] = make_double2(nr / t22, ni / t22);
      }
    }
    // 3. inverse z (exchange first when the output rows are not the input rows)
    if constexpr (!rfft_io_same<NZ>()) {
      __syncthreads();
#pragma unroll
      for (int s = 0; s < NO; ++s)
        if (act && rfft_out_valid<NZ>(t, s)) sh[rfft_out_idx<NZ>(t, s) * TX + c] = a[s];
      __syncthreads();
#pragma unroll
      for (int s = 0; s < NI; ++s)
        if (act && rfft_in_valid<NZ>(t, s)) a[s] = sh[rfft_in_idx<NZ>(t, s) * TX + c];
    }
    rfft<R, NZ, true, TX>(a, t, act, sh + c, tw);
#pragma unroll
    for (int s = 0; s < NO; ++s)
      if (act && rfft_out_valid<NZ>(t, s))
        buf_st<R, AUX>(ROLE == FZ_GHAT ? rg : ru, lw, (unsigned)rfft_out_idx<NZ>(0, s) * rowb, a[s]);
    __syncthreads();
  }
  if (PARS) {
    // block sum: wave sums, then the waves' in order
    double* const red = reinterpret_cast<double*>(sh);
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_down(acc, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = 0.0;
      for (unsigned w = 0; w < (blockDim.x + 63) / 64; ++w) s += red[w];
      part[blockIdx.x] = s * (double)g.P;
    }
  }
}

// ---------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------
int faithful_nonlinear(const Geo& g, const UPar& u, bool diag, const double* st, double* dfd, double* mobd,
                       double* part, long max_blocks, long* nblocks, hipStream_t s) {
  const long grid = std::min<long>(max_blocks, std::max<long>(1, (g.P + kNlBlock - 1) / kNlBlock));
  const size_t shb = sizeof(double) * ((size_t)g.var * kNlBlock + kNlBlock);
  if (diag)
    hipLaunchKernelGGL((k_nl_faithful<true>), dim3((unsigned)grid), dim3(kNlBlock), shb, s, g, u, st, dfd, mobd, part);
  else
    hipLaunchKernelGGL((k_nl_faithful<false>), dim3((unsigned)grid), dim3(kNlBlock), shb, s, g, u, st, dfd, mobd,
                       part);
  *nblocks = grid;
  return 0;
}

template <int ROLE, bool PARS, bool KEEP>
static int zf_launch(const Geo& g, const UPar& u, const KTab& kt, Bank<double> U, Bank<double> D, Bank<double> G,
                     double* part, int f0, int nf, long max_blocks, long* nblocks, hipStream_t s) {
  const double2* tw = twiddle_table<double>(g.nz);
  if (!tw) return fail(PF_EHIP, "twiddle table set-up failed");
  switch (g.nz) {
#define PF_CASE(N)                                                                                      \
  case N: {                                                                                             \
    constexpr int TX = col_tile(N, sizeof(double2));                                                    \
    const long tm = ((long)g.M * g.ny + TX - 1) / TX, tn = ((long)g.ny + TX - 1) / TX;                  \
    long grid = std::min<long>((tm + tn) * nf, max_blocks);                                             \
    /* whole XCD runs of main-block rows (xcd_runs): extra blocks find no tile */                       \
    const long runt = ((long)g.M + TX - 1) / TX, run = 8 * runt;                                        \
    if ((grid + run - 1) / run * run <= max_blocks) grid = (grid + run - 1) / run * run;                \
    hipLaunchKernelGGL((k_zfaithful<N, ROLE, PARS, KEEP>), dim3((unsigned)grid), dim3(TX * plan_T(N)), 0, s, g, u, kt, \
                       U, D, G, part, tw, f0, nf, (unsigned)tm, (unsigned)tn, (unsigned)runt);          \
    if (nblocks) *nblocks = grid;                                                                       \
    return 0;                                                                                           \
  }
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    default: return fail(PF_EINVAL, "unsupported nz");
  }
}

template <bool KEEP>
static int zf_role(int role, bool pars, const Geo& g, const UPar& u, const KTab& kt, Bank<double> U, Bank<double> D,
                   Bank<double> G, double* part, int f0, int nf, long max_blocks, long* nblocks, hipStream_t s) {
  if (role == FZ_ETA)
    return pars ? zf_launch<FZ_ETA, true, KEEP>(g, u, kt, U, D, G, part, f0, nf, max_blocks, nblocks, s)
                : zf_launch<FZ_ETA, false, KEEP>(g, u, kt, U, D, G, part, f0, nf, max_blocks, nblocks, s);
  if (role == FZ_GHAT)
    return pars ? zf_launch<FZ_GHAT, true, KEEP>(g, u, kt, U, D, G, part, f0, nf, max_blocks, nblocks, s)
                : zf_launch<FZ_GHAT, false, KEEP>(g, u, kt, U, D, G, part, f0, nf, max_blocks, nblocks, s);
  return zf_launch<FZ_CMOB, false, KEEP>(g, u, kt, U, D, G, part, f0, nf, max_blocks, nblocks, s);
}

int faithful_z(int role, bool pars, const Geo& g, const UPar& u, const KTab& kt, Bank<double> U, Bank<double> D,
               Bank<double> G, double* part, int f0, int nf, long max_blocks, long* nblocks, hipStream_t s) {
  // the state and derivative banks together
  return bank_stays(2ul * g.F * g.P * sizeof(double))
             ? zf_role<true>(role, pars, g, u, kt, U, D, G, part, f0, nf, max_blocks, nblocks, s)
             : zf_role<false>(role, pars, g, u, kt, U, D, G, part, f0, nf, max_blocks, nblocks, s);
}

}  // namespace pf
