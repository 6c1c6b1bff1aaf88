// Fused kernels of the reduced timestep.
//
// Between steps the work bank W holds every field "x-half-line" state: the full
// spectrum transformed back along z and y but not x.  One step is four kernels:
//   k_xline  : per (y,z) line, all fields: C2R along x -> nonlinear terms ->
//              R2C along x (f_trans normalised), diagnostics of the old state
//   k_ypass  : forward y (main block columns + Nyquist-plane rows)
//   k_zline  : per z column tile: forward z -> semi-implicit update against the
//              carried spectrum S (written back) -> inverse z
//   k_ypass  : inverse y
// so each field's half spectrum crosses HBM 10 times per step (x: 2, y: 2+2,
// z: 4 including S), against 17 for separate transform and pointwise passes.
#pragma once
#include "pf_nl.hpp"
#include "pf_passes.hpp"

namespace pf {

// Deterministic block reductions for any blockDim (multiple of 64).
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}
template <bool MAX> __device__ __forceinline__ double wave_ext(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const double w = __shfl_down(v, o, 64);
    if (MAX ? (w > v) : (w < v)) v = w;
  }
  return v;
}
// red: >= 16 doubles of LDS.  Result valid in thread 0.
__device__ __forceinline__ double bsum(double v, double* red) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int i = 0; i < nw; ++i) s += red[i];
  return s;
}
// Nonlinear terms for NPT = 1 point or NPT = 2 neighbouring points (x = 2k,
// 2k+1: the two halves of one complex LDS element per field), reduced O(var)
// form (gamma block structure of src/var_diff.f90:206-218).  v: field 0 = c,
// fields 1..V = eta, at a stride of fs elements (reals for one point, complex
// for two); the points' arithmetic is independent and interleaved.  Per matrix
// field the derivative
//   eta_i (a_i - 1) + 2 eta_i (s1g (sm - a_i) + s2g av) + cT4m eta_i a_i,  a_i = eta_i^2
// is evaluated as eta_i (alpha a_i + beta) with the point constants
//   alpha = 1 - 2 s1g + cT4m,  beta = 2 (s1g sm + s2g av) - 1,
// one multiply-add and two multiplies per field; the precipitate field's
// derivative likewise as eta_V (gamma av + delta).  The regrouping moves each
// derivative by a few ulp of beta (the derivative enters the update multiplied
// by dt L).  Extremes are tracked in the working precision (exact: they are
// values of the field); the two energy sums in FP64.  The matrix grains' part
// of the bulk energy needs no work per field beyond the sums the derivatives
// use: sum_i (a_i^2 / 4 - a_i / 2) = num / 4 - sm / 2 and
// sum_{i<j} a_i a_j = (sm^2 - num) / 2, with sm = sum a_i, num = sum a_i^2.
template <typename R, int NPT> struct Pts;
template <typename R> struct Pts<R, 1> {
  using T = R;
  static __device__ __forceinline__ R get(const R& v, int) { return v; }
  static __device__ __forceinline__ R make(const R* a) { return a[0]; }
};
template <typename R> struct Pts<R, 2> {
  using T = c2<R>;
  static __device__ __forceinline__ R get(const c2<R>& v, int h) { return h ? v.y : v.x; }
  static __device__ __forceinline__ c2<R> make(const R* a) { return mk<R>(a[0], a[1]); }
};

template <typename R, int NPT, bool DIAG>
__device__ __forceinline__ void nl_points(typename Pts<R, NPT>::T* v, long fs, int V, const UPar& u, R* mo,
                                          double& a_ch, double& a_eta, R& cmax, R& cmin, R& pmin, R& p3) {
  using P = Pts<R, NPT>;
  const R am = (R)u.am, ap = (R)u.ap, cm = (R)u.cm, cp = (R)u.cp, s1g = (R)u.s1g, s2g = (R)u.s2g;
  const int mat = V - 1;
  R con[NPT], sm[NPT], num[NPT], fv[NPT];
  {
    const typename P::T c0 = v[0], f0 = v[V * fs];
#pragma unroll
    for (int h = 0; h < NPT; ++h) {
      con[h] = P::get(c0, h);
      fv[h] = P::get(f0, h);
      sm[h] = num[h] = R(0);
    }
  }
#pragma unroll 2
  for (int i = 1; i <= mat; ++i) {
    const typename P::T f = v[i * fs];
#pragma unroll
    for (int h = 0; h < NPT; ++h) {
      const R fi = P::get(f, h), a = fi * fi;
      sm[h] += a;
      num[h] += a * a;
    }
  }
  R alpha[NPT], beta[NPT], gam[NPT], hm[NPT], hp[NPT], fm[NPT], fpp[NPT], av[NPT], out[NPT];
#pragma unroll
  for (int h = 0; h < NPT; ++h) {
    av[h] = fv[h] * fv[h];
    const R av2 = av[h] * av[h];
    const R d4 = num[h] + av2;
    const R inv_d4 = R(1) / d4;
    hm[h] = num[h] * inv_d4;
    hp[h] = R(1) - hm[h];
    const R dm = con[h] - cm, dp = con[h] - cp;
    fm[h] = am * (dm * dm);
    fpp[h] = ap * (dp * dp);
    out[h] = R(2) * (hm[h] * am * dm + hp[h] * ap * dp);
    const R cT4m = R(4) * (fm[h] - fpp[h]) * (av2 * inv_d4) * inv_d4;
    alpha[h] = (R(1) - R(2) * s1g) + cT4m;
    beta[h] = R(2) * (s1g * sm[h] + s2g * av[h]) - R(1);
    gam[h] = R(1) + R(4) * hm[h] * (fpp[h] - fm[h]) * inv_d4;
  }
  v[0] = P::make(out);
#pragma unroll 2
  for (int i = 1; i <= mat; ++i) {
    const typename P::T f = v[i * fs];
    R o[NPT];
#pragma unroll
    for (int h = 0; h < NPT; ++h) {
      const R fi = P::get(f, h);
      o[h] = fi * (fi * fi * alpha[h] + beta[h]);
    }
    v[i * fs] = P::make(o);
  }
#pragma unroll
  for (int h = 0; h < NPT; ++h) out[h] = fv[h] * (av[h] * gam[h] + (R(2) * s2g * sm[h] - R(1)));
  v[V * fs] = P::make(out);
#pragma unroll
  for (int h = 0; h < NPT; ++h) {
    const R ps = sm[h] + av[h];
    mo[h] = R(2) * (R(1) - ps) * (R)u.Dgb;
    if (DIAG) {
      const R pair = R(0.5) * fma(sm[h], sm[h], -num[h]);
      const R fe = (R(0.25) * num[h] - R(0.5) * sm[h]) + av[h] * (R(0.25) * av[h] - R(0.5)) + s1g * pair +
                   s2g * av[h] * sm[h];
      a_ch += (double)(hm[h] * fm[h] + hp[h] * fpp[h]);
      a_eta += (double)fe;
      if (fv[h] > p3) p3 = fv[h];
      if (con[h] <= cmin) cmin = con[h];
      if (con[h] > cmax) cmax = con[h];
      if (ps < pmin) pmin = ps;
    }
  }
}

// ---------------------------------------------------------------------------
// k_xline: LINES consecutive (y,z) lines of all F fields per iteration.
//   wm, wn : W bank (main block, Nyquist plane); in: x-half lines; out: R2C of
//            the nonlinear derivatives (df_dc, df_dphi_i), divided by P.
//   mobd   : (m - D_mean) per point when mob (input of the mobility chain).
//   XONLY  : mobility-chain variant for one field: C2R, multiply by mobd, R2C.
// One job = one (field, line) x transform, done by T = plan_T(M) threads.  The
// LDS tile is job-major: job j's M complex elements in row j, pitch MP.
//   * A job's T threads are lanes of one wave (xline_wave_jobs), so the transforms'
//     exchanges stay inside the wave and need no block barrier (XF_WAVE).  Element
//     k of a row sits at lds_swz(k) = k + k / 16 (XF_SWZ) and the pitch MP is
//     chosen from a model of the LDS banks over every access pattern of the kernel
//     (exchanges, pairing k with M - k, rows by lanes): the strided exchange
//     accesses of the T lanes and of the 64 / T jobs of a wave then mostly fall
//     on distinct banks.
// Lanes past the jobs skip the transform phases as a whole (one branch, no
// per-slot predicates, no barrier inside).
// A last wave that holds a single job hands it to all its lanes (plan variant
// 3, where the length has one).
// Staging and the final store move whole rows, one or more per wave at a time, and
// do the real <-> half-complex pairing, a lane taking elements k and M - k
// together.  256-point FP32 rows (kXlineTwiddleRegs) skip the final store's row
// pass: each job's 16 threads pair their forward transform's outputs by DPP and
// store them (phase 5).
// The table W_NX^k, k < NX, is copied to LDS once per block for the x transforms
// (length M, stride 2).
// Dynamic LDS: (njobs*MP + NX) complex; the block's diagnostics take six doubles per
// wave of it at the end.
// ---------------------------------------------------------------------------
// Threads per x-line block: FP32 blocks may use 1024 threads, which a 512^3 grid
// with 37 fields needs (37 transforms x 16 threads); FP64 blocks stop at 512
// (640 for 512-point lines, kXlineMaxThreadsN).
template <typename R> constexpr int kXlineMaxThreads = sizeof(R) == 4 ? 1024 : 512;
// FP64 blocks of 512-point lines may use 640 threads (37 fields x 16), 3 waves
// per SIMD at most, which their registers allow.
template <typename R, int NX> constexpr int kXlineMaxThreadsN = (sizeof(R) == 8 && NX >= 512) ? 640 : kXlineMaxThreads<R>;
// Minimum waves per SIMD asked of the register allocator.  FP32: 6 for 128- and
// 160-point lines, which then take up to 79 VGPRs without spills (160^3 x 9: 114 ->
// 102 us against asking for 5); 5 for the others (at 192 points it spills 1 VGPR; 6
// spilled 4, 192^3 x 9 145 -> 185 us; at 256 points 23, 512 -> 694 us); 4 for 512-point lines,
// which keep their last transform pass's twiddles in registers (kXlineTwiddleRegs), at
// most 128 VGPRs, which 1024-thread blocks need anyway.  FP64: 3 (the 256-point kernel takes 167 VGPRs).
template <typename R, int NX>
constexpr int kXlineWavesN = sizeof(R) == 8 ? 3 : NX >= 512 ? 4 : (NX >= 128 && NX < 192) ? 6 : 5;
__host__ __device__ constexpr int xline_T(int M, int cbytes) { return plan_T(M, xline_plan(cbytes)); }
// A job's T threads are lanes of one wave: 64 / T jobs a wave, the lanes past them idle.
__host__ __device__ constexpr int xline_wave_jobs(int M, int cbytes) { return 64 / xline_T(M, cbytes); }
// FP64 rows of 256 points are not padded: a 16-byte access serves 16 lanes a
// cycle, which are one job's T = 16 threads in the exchanges and consecutive
// elements in the row-wise phases, so the rows need no skew; unpadded, 37 fields
// fit one block's LDS (148 KiB of rows).
__host__ __device__ constexpr bool xline_plain_rows(int M, int cbytes) { return cbytes == 16 && M >= 256; }
__host__ __device__ constexpr int xline_xf(int M, int cbytes) {
  return XF_WAVE | (xline_plain_rows(M, cbytes) ? 0 : XF_SWZ);
}
// Row pitch in elements of cbytes bytes: the bank-model choices for FP32
// elements; FP64 rows take the smallest padded pitch (at 512 points they must
// fit 33 rows of 16-byte elements in LDS).
__host__ __device__ constexpr int xline_row_pitch(int M, int cbytes) {
  if (xline_plain_rows(M, cbytes)) return M;
  if (cbytes != 8) return M + M / 16 + 1;
  switch (M) {  // smallest of the bank model's best choices, >= M + M / 16
    case 24: return 26;
    case 32: return 34;
    case 48: return 52;
    case 64: return 72;
    case 96: return 104;
    case 128: return 136;
    case 256: return 272;
    default: return M + M / 16 + 1;
  }
}

// Plan variant 3 (radix 2 at 64 and 128 points, radix 4 at 256): one line done
// by a whole wave.  When njobs = 1 mod 64 / T, the block's last wave carries one
// job on T of its lanes; with this plan its 64 lanes share that job instead and
// the wave issues far fewer transform instructions (at 256^3 x 17, 17 jobs of 8
// threads: x-line kernel 0.577 -> 0.532 ms).
__host__ __device__ constexpr bool xline_has_wide(int M) {
  return M == 64 || M == 128 || M == 256;
}

// One job's x transform with plan V, in place in its LDS row (phases 3 and 5).
// No barrier before the write-back: the last Stockham pass leaves each
// thread's outputs at exactly the elements it loaded as that pass's inputs
// (out_idx = in_idx when j < NB = LS), so no thread overwrites an element
// another thread has yet to read.
// The Nyquist value goes with thread 0, which holds Z_0 = (X_0 + X_M, X_0 - X_M) in
// slot 0: inverse, xn (0 in the other threads) completes it; forward, X_M = Z_0.x -
// Z_0.y goes to *wn (null in the other threads) times scale.
template <typename R, int M, int V, int XF, bool INV, bool TWR = false>
__device__ __forceinline__ void xline_fft(c2<R>* v, c2<R>* col, const c2<R>* shw, int t, R xn, c2<R>* wn, R scale,
                                          const c2<R>* twr = nullptr) {
#pragma unroll
  for (int s = 0; s < kInSlots<M, V>; ++s)
    if (rfft_in_valid<M, V>(t, s)) v[s] = col[lds_swz<XF>(rfft_in_idx<M, V>(t, s))];
  if (INV) v[0] = mk<R>(v[0].x + xn, v[0].y - xn);
  rfft<R, M, INV, 1, V, XF, TWR>(v, t, true, col, shw, 2, 0, twr);
  if (!INV && wn) *wn = mk<R>((v[0].x - v[0].y) * scale, R(0));
#pragma unroll
  for (int s = 0; s < kOutSlots<M, V>; ++s)
    if (rfft_out_valid<M, V>(t, s)) col[lds_swz<XF>(rfft_out_idx<M, V>(t, s))] = v[s];
}

// The real <-> half-complex pairing couples element k of a row with element
// M - k, and the moving waves do it: a lane takes both elements of a pair, from
// HBM when a row is staged and to HBM when it is stored.  Pair p < M / 2 is
// (p, M - p); p = 0 stands for the two self-coupled entries, 0 (with the Nyquist
// value) and M / 2.  A pair's sums and its one twiddle product W_NX^p serve both
// elements (the mirrored element's differ by signs, W_NX^(M-p) = -conj(W_NX^p)),
// about half the arithmetic of two single elements, and every element is read from
// LDS once.  With the pairing one element at a time and vector row addresses, and
// blocks of several line groups: 192^3 x 9 FP32 210 us, 96^3 x 9 30.8, FP64 256^3 x
// 17 1193, 64^3 x 9 26.3; as it is 145, 24.9, 1043 and 15.6 us.
template <int M> __device__ __forceinline__ int xline_partner(int p) { return p ? M - p : M / 2; }
// C2R of a pair: a = X_p, b = X_{M-p} (p = 0: X_0, X_{M/2}) -> Z_p in a, Z_{M-p} in b
// (p = 0: Z_0 without the Nyquist value X_M, which the transform's thread adds, and
// Z_{M/2}).  X_0's imaginary part is not used.
template <typename R> __device__ __forceinline__ void xline_c2r_pair(c2<R>& a, c2<R>& b, c2<R> w, bool p0) {
  const R ay = p0 ? R(0) : a.y, bx = p0 ? R(0) : b.x, by = p0 ? R(0) : b.y;
  const R ar = a.x + bx, ai = ay - by, br = a.x - bx, bi = ay + by;
  const R cr = w.x * br + w.y * bi, ci = w.x * bi - w.y * br;
  a = mk<R>(ar - ci, ai + cr);
  b = mk<R>(p0 ? R(2) * b.x : ar + ci, p0 ? R(-2) * b.y : cr - ai);
}
// R2C of a pair: a = Z_p, b = Z_{M-p} (p = 0: Z_0, Z_{M/2}) -> X_p in a and
// X_{M-p} in b (p = 0: X_0, X_{M/2}); hs = scale / 2.
template <typename R> __device__ __forceinline__ void xline_r2c_pair(c2<R>& a, c2<R>& b, c2<R> w, bool p0, R hs) {
  const R bx = p0 ? a.x : b.x, by = p0 ? a.y : b.y;
  const R ar = a.x + bx, ai = a.y - by, br = a.x - bx, bi = a.y + by;
  const R cr = w.x * br - w.y * bi, ci = w.x * bi + w.y * br;
  const R mx = hs * (ar - ci), my = hs * (-ai - cr);
  a = mk<R>(hs * (ar + ci), hs * (ai - cr));
  b = mk<R>(p0 ? R(2) * hs * b.x : mx, p0 ? R(-2) * hs * b.y : my);
}
// Rows of one field that a wave moves at once: rows of M / 2 pairs, as many of the
// group's LINES as its 64 lanes hold (a power of two; every lane then has a fixed
// row and pair, the rest of the address is scalar).
__host__ __device__ constexpr int xline_rows_at_once(int M, int LINES) {
  int r = 1;
  while (2 * r <= LINES && 2 * r * (M / 2) <= 64) r *= 2;
  return r;
}
// Row groups whose loads a wave keeps in flight: 2; in FP64 3 for 64 and 128 points
// (128^3 x 9: 71.0 -> 67.9 us, 256^3 x 17: 1088 -> 1043 us), where that costs no
// wave per SIMD (at 96 points it did, 192^3 x 9: 338 -> 383 us), and 1 for 256
// points, two pairs a lane (more spilled: 512 x 128 x 128 x 9 348 -> 414 us).
__host__ __device__ constexpr int xline_ahead(int M, int cbytes) {
  return cbytes == 8 ? 2 : (M == 64 || M == 128) ? 3 : M == 256 ? 1 : 2;
}
// 256-point FP32 rows: the last transform pass (radix 16, one butterfly per
// thread) takes its 15 twiddles, the same for every line and both directions,
// from registers loaded once per block rather than from the LDS table.  Those
// blocks hold a CU's LDS alone (37 fields: 85 KB), whose traffic bounds them.
template <typename R, int M>
constexpr bool kXlineTwiddleRegs = M >= 256 && sizeof(R) == 4 && LastPass<M>::Q == 1 && LastPass<M>::LS > 1;
// Lane t of a 16-lane row receives x from lane (16 - t) mod 16 of the same row:
// DPP row_mirror (lane 15 - t) then row_ror:1 (from lane t - 1), register moves
// with no LDS traffic.
__device__ __forceinline__ float dpp_partner16(float x) {
  const int m = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x140, 0xF, 0xF, false);
  const int r = __builtin_amdgcn_update_dpp(0, m, 0x121, 0xF, 0xF, false);
  return __builtin_bit_cast(float, r);
}

// Blocks for ngroups line groups, at most cap: one group each, or an equal number of
// consecutive groups each.  Every block then has its full share but the last; with
// a grid cut at cap itself some blocks carry one group more than others or (ranges of
// ceil(ngroups / cap)) whole XCDs end up without work.  192^3 x 9 in FP32 (18 432
// groups): 220 us cut at 16 384 blocks, 174 us at 8 192, 129 us with one group
// each; 160^3 x 9: 103 us at 8 192, 84 us with one group each; 256^3 x 17 (65 536
// groups): 513 us at 8 192, 506 to 514 us with one or two each.
constexpr long kXlineGroupCap = 65536;
inline long xline_grid(long ngroups, long cap) {
  const long chunk = (ngroups + cap - 1) / cap, grid = (ngroups + chunk - 1) / chunk;
  return grid < 8 ? grid : (grid + 7) / 8 * 8;  // a multiple of 8 for the XCD order
}

// BATCH: ngroups counts the line groups of every member in mt (member m owns
// groups m*gpm .. m*gpm + gpm - 1, gpm = plane / LINES), each taking its banks
// and parameters from its entry; wm, wn, u are unused; no diagnostics.
template <typename R> __device__ __forceinline__ const UPar& member_u(const UPar& u, const Member<R>* mt, long m,
                                                                    bool batch) {
  return batch ? mt[m].u : u;
}

// A block's diagnostics from its threads': wave results side by side in red (LDS, free
// by now), then one thread per value takes the waves' in order.
__device__ __forceinline__ void diag_partials(double ch, double eta, double cmax, double cmin, double pmin, double p3,
                                              double* red, int nw, double* __restrict__ part) {
  const double r0 = wave_sum(ch), r1 = wave_sum(eta);
  const double r2 = wave_ext<true>(cmax), r3 = wave_ext<false>(cmin);
  const double r4 = wave_ext<false>(pmin), r5 = wave_ext<true>(p3);
  if ((threadIdx.x & 63) == 0) {
    double* o = red + 6 * (threadIdx.x >> 6);
    o[0] = r0; o[1] = r1; o[2] = r2; o[3] = r3; o[4] = r4; o[5] = r5;
  }
  __syncthreads();
  const int i = threadIdx.x;
  if (i < 6) {
    double s = red[i];
    for (int w = 1; w < nw; ++w) {
      const double x = red[6 * w + i];
      s = i < 2 ? s + x : (i == 2 || i == 5) ? (x > s ? x : s) : (x < s ? x : s);
    }
    part[(long)blockIdx.x * 6 + i] = s;
  }
}

// KEEP: W stays in cache from pass to pass (bank_stays).
// ROUNDS: the jobs need more threads than a block may have, and the block's waves
// take them in several rounds (in one loop with the common case its registers
// spilled: 256^3 x 17 516 -> 684 us).
// FAITH: the faithful step's x pass (FP64, var <= kNlRegs, LINES * NX threads).  The
// bank has 2F fields.  The real state's R2C goes back to fields 0 .. F-1, the
// derivatives' (in the reference's operation order) to F .. 2F-1.  mob here says that
// the state comes real rather than as x-half lines.  A thread takes its point's values
// into registers, so that the state's rows can be transformed in place before the
// derivatives are written over them: with rows of their own the derivatives left two
// blocks a CU, 256^3 x 17 4.3 ms.  The separate x inverse, pointwise and x forward
// kernels moved seven banks of F, this pass three (a
// step of 256 x 128 x 128 x 17: 1.98 -> 1.61 ms).  At 256 and 512 points the live values
// take 208 and 200 VGPRs, two waves per SIMD; at three waves it spills 38 to 40 VGPRs a
// lane at 24 points, 8 to 14 at 96, 2 at 48 and 160, none elsewhere.
template <typename R, int NX, int LINES, bool XONLY, bool BATCH = false, bool KEEP = false, bool ROUNDS = false,
          bool FAITH = false>
__global__ void __launch_bounds__((FAITH ? 512 : kXlineMaxThreadsN<R, NX>))
__attribute__((amdgpu_waves_per_eu(FAITH && NX >= 256 ? 2 : kXlineWavesN<R, NX>)))
k_xline(Geo g, UPar u, c2<R>* __restrict__ wm, c2<R>* __restrict__ wn, R* __restrict__ mobd,
        const c2<R>* __restrict__ tw, double* __restrict__ part, long ngroups, int diag, int mob,
        const Member<R>* __restrict__ mt) {
  constexpr int M = NX / 2, XV = xline_plan(sizeof(c2<R>)), T = plan_T(M, XV);
  constexpr int MP = xline_row_pitch(M, sizeof(c2<R>)), XF = xline_xf(M, sizeof(c2<R>));
  constexpr bool HAVEW = !FAITH && xline_has_wide(M);
  // the wide plan's variant (3) and threads; the T-thread plan stands in when
  // this length has no wide plan, and that branch is never taken then
  constexpr int WV = HAVEW ? 3 : XV, TW = plan_T(M, WV), JW = xline_wave_jobs(M, sizeof(c2<R>));
  static_assert(last_pass_in_place<M, XV>(), "the write-backs after the x transforms rely on it");
  extern __shared__ unsigned char smem[];
  const int F = XONLY ? 1 : g.F;
  const int njobs = F * LINES;
  c2<R>* sh = reinterpret_cast<c2<R>*>(smem);
  constexpr bool TR = kXlineTwiddleRegs<R, M>;
  c2<R>* shw = sh + (long)njobs * MP;  // W_NX^k, k < NX
  const int nt = blockDim.x, nw = nt >> 6;
  constexpr int H = M / 2, PPL = (H + 63) / 64;  // pairs of a row, and per lane
  constexpr int RP = xline_rows_at_once(M, LINES), NA = xline_ahead(M, sizeof(c2<R>));
  const int npieces = F * (LINES / RP);
  for (int k = threadIdx.x; k < NX; k += nt) shw[k] = tw[k];
  if constexpr (TR) __syncthreads();
  c2<R> twr[TR ? LastPass<M>::r - 1 : 1];
  if constexpr (TR) last_pass_twiddles<R, M>(twr, (threadIdx.x & 63) % T, shw, 2);
  const R scale = (R)u.invP;
  double a_ch = 0.0, a_eta = 0.0;
  R cmax = 0, cmin = 1, pmin = 1, p3 = 0;
  c2<R> v[plan_E(M, XV) > plan_E(M, WV) ? plan_E(M, XV) : plan_E(M, WV)];

  // each block takes the same number of consecutive line groups (xline_grid)
  const unsigned lb = (unsigned)xcd_block(blockIdx.x, gridDim.x);
  const unsigned chunk = ((unsigned)ngroups + gridDim.x - 1) / gridDim.x;
  const unsigned lg0 = lb * chunk, lg1 = lg0 + chunk < (unsigned)ngroups ? lg0 + chunk : (unsigned)ngroups;
  for (long lg = lg0; lg < lg1; ++lg) {
    // Per-thread indices are recomputed each iteration from an opaque copy of
    // the thread id: hoisted, the addresses derived from them stayed live across
    // the loop (and the transforms' twiddles, read from global memory, too),
    // 126 VGPRs at 256^3 x 17; recomputed, with the twiddles from LDS, 90.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    // the wave's number, uniform: the rows a wave moves then have scalar addresses
    const int wv = __builtin_amdgcn_readfirstlane(tid) >> 6;
    const int t = lane % T;
    const bool lact = 64 % T == 0 || lane < JW * T;
    // the lone job of the last wave (njobs = 1 mod 64 / T) goes to the whole
    // wave; the condition is uniform over the wave (a scalar branch)
    const bool wide_any = HAVEW && njobs % JW == 1;
    const auto is_wide = [&](int jr) { return wide_any && jr + wv * JW == njobs - 1; };
    long L0 = lg * LINES, m = 0;
    c2<R>* wmm = wm;
    c2<R>* wnn = wn;
    if constexpr (BATCH) {
      const long gpm = g.plane / LINES;
      m = lg / gpm;
      L0 = (lg - m * gpm) * LINES;
      wmm = mt[m].Wm;
      wnn = mt[m].Wn;
    }
    const UPar& uu = member_u<R>(u, mt, m, BATCH);
    // the Nyquist entry of this thread's job in round jr (thread 0 of a job takes it)
    const auto nyq = [&](int jr, int ln, int lt) -> c2<R>* {
      const bool wide = is_wide(jr);
      const int jn = wide ? njobs - 1 : jr + wv * JW + ln / T, fn = jn / LINES;
      const bool has = wide ? ln == 0 : lact && lt == 0 && jn < njobs;
      return has ? wnn + (long)fn * g.plane + L0 + (jn - fn * LINES) : nullptr;
    };
    R xn = R(0);
    if (const c2<R>* p = nyq(0, lane, t)) xn = p->x;
    // this lane's row within a wave's row group and its pairs' elements
    const int sub = H >= 64 ? 0 : lane / H, p0 = H >= 64 ? lane : lane - sub * H;
    const bool mine = H >= 64 || sub < RP;
    // 1. half lines of every field -> LDS rows, with the C2R pre-processing: wave w
    //    stages row groups w, w + nw, ... (coalesced along k, and along M - k in
    //    descending order), NA of them in flight
    const bool real = FAITH && mob;
    c2<R> w[PPL];  // a lane's pairs, and so their twiddles, are the same in every row
#pragma unroll
    for (int i = 0; i < PPL; ++i) w[i] = tw[p0 + 64 * i];
    if (real) {
      for (int f = wv; f < F; f += nw) {
        const c2<R>* src = wmm + (long)f * g.hmain + L0 * M;
        for (int e = lane; e < LINES * M; e += 64)
          sh[(f * LINES + e / M) * MP + lds_swz<XF>(e % M)] = src[e];
      }
    } else
    for (int j0 = wv; j0 < npieces; j0 += NA * nw) {
      c2<R> ta[NA][PPL], tb[NA][PPL];
#pragma unroll
      for (int r = 0; r < NA; ++r) {
        const int j = j0 + r * nw;
        if (j < npieces) {
          const int f = j / (LINES / RP), l = (j - f * (LINES / RP)) * RP;
          const c2<R>* src = wmm + (long)f * g.hmain + (L0 + l) * M;
          if (mine) {
#pragma unroll
            for (int i = 0; i < PPL; ++i) {
              const int p = p0 + 64 * i;
              const c2<R>*a = src + (sub * M + p), *b = src + (sub * M + xline_partner<M>(p));
              ta[r][i] = KEEP ? *a : ld_nt<R>(a);
              tb[r][i] = KEEP ? *b : ld_nt<R>(b);
            }
          }
        }
      }
#pragma unroll
      for (int r = 0; r < NA; ++r) {
        const int j = j0 + r * nw;
        if (j < npieces && mine) {
          c2<R>* rw = sh + (j * RP + sub) * MP;
#pragma unroll
          for (int i = 0; i < PPL; ++i) {
            const int p = p0 + 64 * i;
            xline_c2r_pair<R>(ta[r][i], tb[r][i], w[i], p == 0);
            rw[lds_swz<XF>(p)] = ta[r][i];
            rw[lds_swz<XF>(xline_partner<M>(p))] = tb[r][i];
          }
        }
      }
    }
    __syncthreads();
    // 2-3. inverse x transform of each job; real pairs z[n] = (x[2n], x[2n+1]).
    if (!real)
    for (int jr = 0; jr < (ROUNDS ? njobs : 1); jr += ROUNDS ? nw * JW : 1) {
      const int job = jr + wv * JW + lane / T;
      if (jr > 0) {
        const c2<R>* p = nyq(jr, lane, t);
        xn = p ? p->x : R(0);
      }
      if (is_wide(jr)) {
        if (TW == 64 || lane < TW)
          xline_fft<R, M, WV, XF, true>(v, sh + (njobs - 1) * MP, shw, lane, xn, nullptr, scale);
      } else if (lact && job < njobs) {
        xline_fft<R, M, XV, XF, true, TR>(v, sh + job * MP, shw, t, xn, nullptr, scale, twr);
      }
    }
    __syncthreads();
    // 4. pointwise: point x of line l is component x%2 of element x/2 of row
    //    f*LINES + l.  When the group has more points than the block has threads
    //    (256 points, 192 threads at 256^3 x 17), each thread takes the two
    //    points of one element: one pass instead of two for the first wave
    //    (measured 0.645 -> 0.616 ms); otherwise one point per thread (pairs
    //    measured 4% slower at 128^3, where the points fit one pass anyway).
    R pf[FAITH ? kNlRegs : 1], pc = R(0), pv = R(0);  // FAITH: the thread's point
    R* pt = nullptr;
    if constexpr (FAITH) {
      if (tid < LINES * NX) {
        constexpr long fs = 2L * LINES * MP;
        const int l = tid / NX, x = tid - l * NX;
        pt = reinterpret_cast<R*>(sh) + 2L * ((long)l * MP + lds_swz<XF>(x >> 1)) + (x & 1);
        pc = pt[0];
        pv = pt[g.var * fs];
#pragma unroll
        for (int i = 0; i < kNlRegs; ++i) pf[i] = i < g.var - 1 ? pt[(i + 1) * fs] : R(0);
      }
    } else if (!XONLY && LINES * NX > nt) {
      constexpr long fs = (long)LINES * MP;  // field stride in complex elements
      for (int p = tid; p < LINES * M; p += nt) {
        const int l = p / M, k = p - l * M;
        c2<R>* vv = sh + (long)l * MP + lds_swz<XF>(k);
        const long gp = (L0 + l) * NX + 2 * k;  // point index within a field
        R mo[2];
        if (diag) nl_points<R, 2, true>(vv, fs, g.var, uu, mo, a_ch, a_eta, cmax, cmin, pmin, p3);
        else nl_points<R, 2, false>(vv, fs, g.var, uu, mo, a_ch, a_eta, cmax, cmin, pmin, p3);
        if (mob) {
          mobd[gp] = mo[0];
          mobd[gp + 1] = mo[1];
        }
      }
    } else {
      R* rl = reinterpret_cast<R*>(sh);
      constexpr long fs = 2L * LINES * MP;  // field stride in reals
      for (int p = tid; p < LINES * NX; p += nt) {
        const int l = p / NX, x = p - l * NX;
        R* vv = rl + 2L * ((long)l * MP + lds_swz<XF>(x >> 1)) + (x & 1);
        const long gp = (L0 + l) * NX + x;
        if (XONLY) {
          vv[0] = vv[0] * mobd[gp];
        } else {
          R mo[1];
          if (diag) nl_points<R, 1, true>(vv, fs, g.var, uu, mo, a_ch, a_eta, cmax, cmin, pmin, p3);
          else nl_points<R, 1, false>(vv, fs, g.var, uu, mo, a_ch, a_eta, cmax, cmin, pmin, p3);
          if (mob) mobd[gp] = mo[0];
        }
      }
    }
    __syncthreads();
    const auto forward = [&](const int half) __attribute__((always_inline)) {
      // 5. forward x transform of each job.  With TR (256-point FP32 rows, 16
      //    threads a job, one 16-lane DPP row each) a job's threads also do its R2C
      //    post-processing and store: after the last pass thread t holds
      //    Z[t + 16 s] in slot s, whose partner Z[M - t - 16 s] is slot 15 - s of
      //    thread 16 - t (for t = 0: its own slot (16 - s) mod 16), so the pairs
      //    come by DPP instead of a write-back and a second read of the row (512^3
      //    x 37: x line 13.5-13.8 -> 13.0-13.1 ms).  The lone wide job, if any,
      //    still goes through its row and phase 6.
      for (int jr = 0; jr < (ROUNDS ? njobs : 1); jr += ROUNDS ? nw * JW : 1) {
        // recomputed rather than kept in registers through the phases between
        int tn = threadIdx.x;
        asm volatile("" : "+v"(tn));
        const int ln = tn & 63, lt = ln % T, job = jr + wv * JW + ln / T;
        c2<R>* wnj = nyq(jr, ln, lt);
        if (FAITH && half && wnj) wnj += (long)F * g.plane;
        if (is_wide(jr)) {
          if (TW == 64 || ln < TW)
            xline_fft<R, M, WV, XF, false>(v, sh + (njobs - 1) * MP, shw, ln, R(0), wnj, scale);
        } else if (lact && job < njobs) {
          c2<R>* const col = sh + job * MP;
          if constexpr (TR) {
            static_assert(T == 16 && kInSlots<M> == 16 && kOutSlots<M> == 16, "16 threads, 16 slots a job");
#pragma unroll
            for (int s = 0; s < 16; ++s) v[s] = col[lds_swz<XF>(rfft_in_idx<M>(lt, s))];
            rfft<R, M, false, 1, 0, XF, true>(v, lt, true, col, shw, 2, 0, twr);
            const int f = job / LINES, l = job - f * LINES;
            c2<R>* dst = wmm + (long)f * g.hmain + (L0 + l) * M;
            const R hs = R(0.5) * scale;
#pragma unroll
            for (int s = 0; s < 16; ++s) {
              const int k = rfft_out_idx<M>(lt, s);  // t + 16 s
              const c2<R> src = v[15 - s];
              c2<R> pr = mk<R>(dpp_partner16(src.x), dpp_partner16(src.y));
              if (lt == 0) pr = v[(16 - s) % 16];
              const c2<R> x = r2c_post<R>(v[s], pr, shw[k], hs);
              if constexpr (KEEP) dst[k] = x;
              else st_nt<R>(dst + k, x);
            }
            if (lt == 0) *wnj = mk<R>((v[0].x - v[0].y) * scale, R(0));
          } else {
            xline_fft<R, M, XV, XF, false, TR>(v, col, shw, lt, R(0), wnj, scale, twr);
          }
        }
      }
      __syncthreads();
      // 6. R2C post-processing and store, the row groups and pairs of 1 (with TR only
      //    the wide job's row)
      const R hs = R(0.5) * scale;
#pragma unroll
      for (int i = 0; i < PPL; ++i) w[i] = shw[p0 + 64 * i];
      for (int j = wv; j < npieces; j += nw) {
        if (TR && !(wide_any && j == njobs - 1)) continue;
        const int f = j / (LINES / RP), l = (j - f * (LINES / RP)) * RP;
        c2<R>* dst = wmm + (long)(FAITH && half ? F + f : f) * g.hmain + (L0 + l) * M;
        const c2<R>* rw = sh + (j * RP + sub) * MP;
        if (!mine) continue;
#pragma unroll
        for (int i = 0; i < PPL; ++i) {
          const int p = p0 + 64 * i, q = xline_partner<M>(p);
          c2<R> a = rw[lds_swz<XF>(p)], b = rw[lds_swz<XF>(q)];
          xline_r2c_pair<R>(a, b, w[i], p == 0, hs);
          if constexpr (KEEP) {
            dst[sub * M + p] = a;
            dst[sub * M + q] = b;
          } else {
            st_nt<R>(dst + (sub * M + p), a);
            st_nt<R>(dst + (sub * M + q), b);
          }
        }
      }
    };
    forward(0);
    if constexpr (FAITH) {
      __syncthreads();
      if (pt) {
        // not before the state's transforms: the products of these would be held too
        asm volatile("" : "+v"(pc), "+v"(pv));
#pragma unroll
        for (int i = 0; i < kNlRegs; ++i) asm volatile("" : "+v"(pf[i]));
        constexpr long fs = 2L * LINES * MP;
        const auto put = [&](int i, R y) { pt[i * fs] = y; };
        R mo;
        if (diag) nl_point_regs<true>(uu, g.var, pc, pf, pv, put, mo, a_ch, a_eta, cmax, cmin, pmin, p3);
        else nl_point_regs<false>(uu, g.var, pc, pf, pv, put, mo, a_ch, a_eta, cmax, cmin, pmin, p3);
        mobd[L0 * NX + (long)threadIdx.x] = mo;
      }
      __syncthreads();
      forward(1);
    }
    __syncthreads();
  }
  if (!XONLY && diag) {
    diag_partials(a_ch, a_eta, (double)cmax, (double)cmin, (double)pmin, (double)p3, reinterpret_cast<double*>(smem),
                  nw, part);
  }
}

// ---------------------------------------------------------------------------
// k_zline: forward z -> update -> inverse z on column tiles of each field.
// ROLE_REG : c (D_gb = 0 form) and eta updates; W -> S, W
// ROLE_GHAT: c only; W_c -> f^ (stored to X) and g^ = kf_sum f^ - kappa_c c^ k_cube,
//            inverse z of g^ -> Y
// ROLE_CMOB: c only; h^ from Y (forward z) with f^ from X -> S_c, W_c
// The spectrum values a thread holds after the forward transform are updated in
// registers (S read and written at the same rows); when the transform's output
// rows differ from its input rows an LDS exchange precedes the inverse.
// S is stored in the kernel's own tile order: tile tt of field f (tt < tm: main
// block columns tt*TX .., else Nyquist-plane columns) is NZ rows of TX complex,
// contiguous, at S.main + ((f*(tm+tn) + tt)*NZ + z)*TX + column (Geo::stx, stm,
// stpf describe it).  Every tile of S is then one contiguous 32 KiB (FP32,
// NZ = 256) block rather than NZ row segments one z plane apart.  At 256^3 x 17
// a copy of the pass's data movement alone went 0.99 -> 0.87 ms; the pass
// itself, with the buffer addressing below, 0.962 -> 0.929 ms.
// The wavenumbers and the update coefficients are evaluated in FP64 in both
// precisions: in FP32 a rounded coefficient A = 1/(1 + dt M kappa k^4) would
// bias every step the same way, and over 1000 steps of a slowly decaying mode
// that bias grows linearly (measured 1.5e-4 max error in c at 256^3 x 17,
// against rounding of the products alone, which averages out).
// ---------------------------------------------------------------------------
enum { ROLE_REG = 0, ROLE_GHAT = 1, ROLE_CMOB = 2 };

// 1/x in FP64 for x in [1, 2^60): hardware reciprocal estimate and two Newton
// steps (each doubles the correct bits), within a few ulp of the quotient.
__device__ __forceinline__ double recip_fast(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = r * (2.0 - x * r);
  return r * (2.0 - x * r);
}

// Minimum waves per SIMD asked of the register allocator: 3 for FP32 plans with
// up to 16 complex values per thread, 2 for plans holding more (E > 16) and for
// FP64.  At 256 the FP32 update takes 165 VGPRs (3 waves) with no spills;
// capped at 4 waves it spilled 6-25 registers per lane and ran 16% slower.
template <typename R, bool PARSEVAL, int E = 16> constexpr int kZlineWaves = (sizeof(R) == 4 && E <= 16) ? 3 : 2;
// 512-point FP32 columns with the 32-thread plans (V = 1, 2: 512-thread blocks,
// 64 KiB of LDS): capped at 128 VGPRs (4 waves per SIMD) two blocks share a CU,
// one loading while the other transforms.  They spill 11-15 VGPRs per lane that
// way and still take 16.3-16.5 ms per update pass at 512^3 x 37, against
// 21.0-22.3 ms uncapped (one block per CU) and 20.9 ms for the default plan's
// 1 024-thread blocks.
template <typename R, int NZ, int V, bool PARSEVAL>
constexpr int kZlineWavesN = (sizeof(R) == 4 && NZ >= 512 && V > 0) ? 4 : kZlineWaves<R, PARSEVAL, plan_E(NZ, V)>;

// The update coefficients of one parameter set, FP64.
struct ZCo {
  double Dk, Ddt, Lkd, Ldt, dt, kc, kphi;
};
__device__ __forceinline__ ZCo zco(const UPar& u) {
  return ZCo{(u.D * u.dt) * u.kc, u.D * u.dt, (u.L * u.kphi) * u.dt, u.L * u.dt, u.dt, u.kc, u.kphi};
}

// KEEP: cache policy (bank_stays): 0 = every bank streamed, 1 = W (and X, Y) stays,
// S streamed, 2 = both stay.  A template parameter: with the accesses of both
// policies behind a uniform branch the kernel spilled.
// BATCH (ROLE_REG only): the fields f0 .. f0 + nf - 1 run over every member in
// mt, g.F per member, each with its own S, W, k = 0 modes and parameters; S, W
// and dc64 are unused.
template <typename R, int NZ, int ROLE, bool DC64, bool PARSEVAL, bool BATCH = false, int V = 0, int KEEP = 0>
__global__ void __launch_bounds__(col_tile(NZ, sizeof(c2<R>)) * plan_T(NZ, V))
__attribute__((amdgpu_waves_per_eu(kZlineWavesN<R, NZ, V, PARSEVAL>)))
k_zline(Geo g, UPar u, KTab kt, Bank<R> S, Bank<R> W, Bank<R> X, Bank<R> Y,
        double* __restrict__ dc64, double* __restrict__ part, const c2<R>* __restrict__ tw, int f0, int nf,
        long tm, long tn, long run_tiles, const Member<R>* __restrict__ mt) {
  static_assert(!BATCH || ROLE == ROLE_REG, "batched members step without the mobility chain");
  constexpr int TX = col_tile(NZ, sizeof(c2<R>));
  constexpr int NI = kInSlots<NZ, V>, NO = kOutSlots<NZ, V>, E = plan_E(NZ, V);
  constexpr unsigned CB = sizeof(c2<R>);
  constexpr int AUXW = KEEP ? 0 : kBufNT, AUXS = KEEP == 2 ? 0 : kBufNT;
  static_assert(last_pass_in_place<NZ, V>(), "slot rows of the last pass are t + a per-slot constant");
  // the exchange tile (up to 64 KiB), which after the tile loop holds the
  // block reduction's 16 doubles
  constexpr int SHN = (plan_np(NZ, V) > 1) ? NZ * TX : 1;
  __shared__ c2<R> sh[SHN * sizeof(c2<R>) >= 16 * sizeof(double) ? SHN : 16 * sizeof(double) / sizeof(c2<R>)];
  double* const red = reinterpret_cast<double*>(sh);
  const long tpf = tm + tn;
  const long total = (long)nf * tpf;
  const int c = threadIdx.x % TX, t = threadIdx.x / TX;
  const ZCo z0c = zco(u);
  double acc = 0.0;
  c2<R> v[E];
  c2<R> sv[NO];
  c2<R> xv[(ROLE == ROLE_CMOB) ? NO : 1];
  const long tile0 = xcd_runs(blockIdx.x, gridDim.x, run_tiles);
  for (long tile = tile0; tile < total; tile += gridDim.x) {
    int f = f0 + (int)(tile / tpf);
    Bank<R> Sb = S, Wb = W;
    double* dcb = dc64;
    ZCo zc = z0c;
    if constexpr (BATCH) {
      const long m = f / g.F;
      f -= (int)(m * g.F);
      Sb = Bank<R>{mt[m].S, nullptr};
      Wb = Bank<R>{mt[m].Wm, mt[m].Wn};
      dcb = mt[m].dc64;
      zc = zco(mt[m].u);
    }
    const long tt = tile % tpf;
    const bool isn = tt >= tm;
    const long Wd = isn ? (long)g.ny : (long)g.M * g.ny;
    const long col0 = (isn ? tt - tm : tt) * TX;
    const int ncol = (int)((Wd - col0) < TX ? (Wd - col0) : TX);
    const bool act = c < ncol;
    // Buffer descriptors on the tile's first column (block-uniform): the
    // natural-layout banks W, X, Y (z rows Wd columns apart; X, Y hold field c
    // only) and the tile of S.  A thread's row of slot s is its own t plus a
    // per-slot constant (first pass: in_idx; last pass, in place: out_idx), so
    // every access is one lane offset plus a uniform one.
    const unsigned rowb = (unsigned)Wd * CB, nb = (unsigned)NZ * rowb;
    const BufRes rw = buf_res((isn ? Wb.nyq : Wb.main) + (isn ? (long)f * g.plane : (long)f * g.hmain) + col0, nb);
    const BufRes rx = buf_res((isn ? X.nyq : X.main) + col0, nb);
    const BufRes ry = buf_res((isn ? Y.nyq : Y.main) + col0, nb);
    const BufRes rs = buf_res(Sb.main + ((long)f * tpf + tt) * ((long)NZ * TX), (unsigned)(NZ * TX) * CB);
    const unsigned lw = ((unsigned)t * (unsigned)Wd + (unsigned)c) * CB;  // natural layout
    const unsigned ls = (unsigned)threadIdx.x * CB;                        // S tile: row t, column c
    // 1. all loads of the tile at once: transform input, spectrum (and f^) at the output rows
#pragma unroll
    for (int s = 0; s < NI; ++s)
      if (act && rfft_in_valid<NZ, V>(t, s))
        v[s] = buf_ld<R, AUXW>((ROLE == ROLE_CMOB) ? ry : rw, lw, (unsigned)rfft_in_idx<NZ, V>(0, s) * rowb);
#pragma unroll
    for (int s = 0; s < NO; ++s)
      if (act && rfft_out_valid<NZ, V>(t, s)) {
        sv[s] = buf_ld<R, AUXS>(rs, ls, (unsigned)(rfft_out_idx<NZ, V>(0, s) * TX) * CB);
        if constexpr (ROLE == ROLE_CMOB) xv[s] = buf_ld<R, 0>(rx, lw, (unsigned)rfft_out_idx<NZ, V>(0, s) * rowb);
      }
    const long col = act ? col0 + c : 0;  // a padding column's would be past the tables' end
    const int kx = isn ? g.M : (int)(col % g.M);
    const int ky = isn ? (int)col : (int)(col / g.M);
    const KCol<double> kc = kcol<double>(kt, kx, ky);
    const double kap = (f == 0) ? zc.kc : zc.kphi;
    // The z wavenumbers of a thread's rows are the same for every tile; an
    // opaque copy of t keeps the compiler from hoisting all of them (2 doubles
    // per slot) out of the tile loop into registers, recomputing them instead.
    int tz = t;
    asm volatile("" : "+v"(tz));
    // 2. forward z, update in registers
    rfft<R, NZ, false, TX, V>(v, t, act, sh + c, tw);
#pragma unroll
    for (int s = 0; s < NO; ++s) {
      if (!(act && rfft_out_valid<NZ, V>(t, s))) continue;
      const int e = rfft_out_idx<NZ, V>(t, s);
      const KCoefR<double> k = kcoef_z(kc, rfft_out_idx<NZ, V>(tz, s), NZ, kt.uz);
      const c2<R> w = v[s];
      c2<R> sn;
      if constexpr (ROLE == ROLE_GHAT) {
        const c2<R> ch = sv[s];
        buf_st<R, 0>(rx, lw, (unsigned)rfft_out_idx<NZ, V>(0, s) * rowb, w);  // f^
        sn = mk<R>((R)(-(k.s1 * w.y) + zc.kc * ch.y * k.k3), (R)(k.s1 * w.x - zc.kc * ch.x * k.k3));
      } else {
        const c2<R> s0 = sv[s];
        // A = 1/den multiplies the whole state each step; B (and Cc) the step's
        // increment
        const double den = (f == 0) ? 1.0 + zc.Dk * k.k4 : 1.0 - zc.Lkd * k.k2;
        if constexpr (sizeof(R) == 8) {
          const double A = 1.0 / den;
          const double B = (f == 0) ? (zc.Ddt * k.k2) * A : -zc.Ldt * A;
          if constexpr (ROLE == ROLE_CMOB) {
            const c2<R> fh = xv[s];
            const double Cc = (zc.dt * k.s1) * A;
            sn = mk<R>(A * s0.x + B * fh.x - Cc * w.y, A * s0.y + B * fh.y + Cc * w.x);
          } else {
            sn = mk<R>(A * s0.x + B * w.x, A * s0.y + B * w.y);
          }
        } else {
          // FP32 state: A carried as an unevaluated sum hi + lo of two floats, so
          // the only per-step error on the state is the rounding of the products
          const double A = recip_fast(den);
          const float Ah = (float)A, Al = (float)(A - (double)Ah);
          const float B = (float)((f == 0) ? (zc.Ddt * k.k2) * A : -zc.Ldt * A);
          float ix = B * (float)w.x, iy = B * (float)w.y;
          if constexpr (ROLE == ROLE_CMOB) {
            const c2<R> fh = xv[s];
            const float Cc = (float)((zc.dt * k.s1) * A);
            ix = B * fh.x - Cc * w.y;
            iy = B * fh.y + Cc * w.x;
          }
          sn = mk<R>(fmaf(Ah, s0.x, fmaf(Al, s0.x, ix)), fmaf(Ah, s0.y, fmaf(Al, s0.y, iy)));
        }
        if (DC64 && kx == 0 && ky == 0 && e == 0) {
          if (f != 0) dcb[f] = dcb[f] - zc.Ldt * (double)w.x;
          sn = mk<R>((R)dcb[f], R(0));
        }
        buf_st<R>(rs, ls, (unsigned)(rfft_out_idx<NZ, V>(0, s) * TX) * CB, sn);

      }
      v[s] = sn;
    }
    if (PARSEVAL && ROLE != ROLE_GHAT) {
      // Parseval terms of the new spectrum, in a pass of their own after the
      // update (fewer registers live at once): |kf'|^2 = (x,y part) + azp^2,
      // the column part applied once per tile
      R pa1 = R(0), pa2 = R(0);
#pragma unroll
      for (int s = 0; s < NO; ++s) {
        if (!(act && rfft_out_valid<NZ, V>(t, s))) continue;
        const R m2 = v[s].x * v[s].x + v[s].y * v[s].y;
        const int ez = rfft_out_idx<NZ, V>(tz, s);
        const R zp = (2 * ez == NZ) ? R(0) : (R)az_of(ez, NZ, kt.uz);  // a'_z: a_z zeroed at Nyquist
        pa1 += m2;
        pa2 += zp * zp * m2;
      }
      const double wgt = (kx == 0 || kx == g.M) ? 1.0 : 2.0;
      acc += (0.5 * kap) * wgt * (kc.kp2 * (double)pa1 + (double)pa2);
    }
    // 3. inverse z (exchange first when the output rows are not the input rows)
    if constexpr (!rfft_io_same<NZ, V>()) {
      __syncthreads();
#pragma unroll
      for (int s = 0; s < NO; ++s)
        if (act && rfft_out_valid<NZ, V>(t, s)) sh[rfft_out_idx<NZ, V>(t, s) * TX + c] = v[s];
      __syncthreads();
#pragma unroll
      for (int s = 0; s < NI; ++s)
        if (act && rfft_in_valid<NZ, V>(t, s)) v[s] = sh[rfft_in_idx<NZ, V>(t, s) * TX + c];
    }
    rfft<R, NZ, true, TX, V>(v, t, act, sh + c, tw);
#pragma unroll
    for (int s = 0; s < NO; ++s)
      if (act && rfft_out_valid<NZ, V>(t, s))
        buf_st<R, AUXW>((ROLE == ROLE_GHAT) ? ry : rw, lw, (unsigned)rfft_out_idx<NZ, V>(0, s) * rowb, v[s]);
    __syncthreads();
  }
  if (PARSEVAL) {
    const double s = bsum(acc, red);
    if (threadIdx.x == 0) part[blockIdx.x] = s * (double)g.P;
  }
}

}  // namespace pf
