// Axis-pass kernels of the 3-D real<->half-complex transform.
//
// Layout of one field ("split-Nyquist half spectrum"):
//   main block  S[kz][ky][kx], kx in [0, M), M = NX/2, kx fastest   (M*NY*NZ complex)
//   Nyquist     Q[kz][ky]      for kx = M, ky fastest               (NY*NZ complex)
// The main block occupies exactly the bytes of the real field (NX*NY*NZ reals),
// so R2C and C2R run in place; the Nyquist plane lives in its own array.  With
// the odd kx = M column moved out, every y- and z-pass access is a run of whole
// cache lines.
//
// Batches of fields are contiguous: field f's main block starts at f*M*NY*NZ and
// its Nyquist plane at f*NY*NZ, so "lines" of the x pass are numbered
// L = y + NY*(z + NZ*f) across the batch.
//
// Transforms use the register-resident Stockham of pf_fft2.hpp: pass-0 inputs
// are loaded from HBM straight into registers and last-pass outputs are stored
// from registers; LDS is only used for the transposes between passes (and, in
// the x pass, for the real<->half-complex pairing of k and M-k).
#pragma once
#include "pf_fft2.hpp"

namespace pf {

constexpr int kBlock = 256;

// columns per tile of a column pass: a power of two from 16 to 64 (every row
// segment a whole number of 128-byte lines), block of <= ~256 threads, exchange
// tile <= 64 KiB.  (Lengths 96, 160, 192 have T = 6, 10, 12 threads per column;
// 256/T would give 42, 25, 21 columns and misaligned segments, which ran the
// 192^3 z-line at 1.8 TB/s.)
__host__ __device__ constexpr int col_tile(int N, int cbytes) {
  const int want = kBlock / plan_T(N);
  int tx = 16;
  while (tx * 2 <= want && tx < 64) tx *= 2;
  while (tx > 1 && N * tx * cbytes > 65536) tx /= 2;
  return tx;
}
// lines per block of a contiguous-line pass
__host__ __device__ constexpr int lines_per_block(int N) {
  return (kBlock / plan_T(N)) > 0 ? (kBlock / plan_T(N)) : 1;
}

// Map physical block ids to logical ones so that each XCD (blocks are dealt to
// the 8 XCDs round-robin) works on a contiguous range of tiles or lines.  The x
// line kernel's neighbouring lines then share that XCD's L2 for the Nyquist
// entries, and a column pass's neighbouring tiles (the 128-byte pieces of the
// same rows) are read by one XCD at about the same time: measured at 256^3 x 17,
// column passes 3-7% faster.  (The z-line kernel measured 1.05 against 1.34 ms
// with this remap; it uses xcd_runs below.)
__device__ __forceinline__ long xcd_block(long b, long nb) {
  if (nb % 8) return b;
  return (b % 8) * (nb / 8) + b / 8;
}

// The same in runs of G: XCD x takes the blocks x*G .. x*G + G - 1 of every 8*G
// (unchanged when the grid is not a multiple of 8*G).  The z-line kernel uses
// runs of one main-block row (M / TX tiles), so each XCD reads whole 1 KiB rows
// of a z plane: measured at 256^3 x 17, 1.055 -> 1.003 ms per launch (runs of
// 8-32 tiles alike; 256 tiles 1.036, one contiguous range per XCD 1.34).
__device__ __forceinline__ long xcd_runs(long b, long nb, long G) {
  if (G < 1 || nb % (8 * G)) return b;
  const long x = b % 8, i = b / 8;
  return (i / G) * (8 * G) + x * G + i % G;
}

// Lines per block of the x passes (k_x_r2c, k_x_c2r).  FP64:
// blocks of one wave (e.g. 8 lines of 8 threads at NX = 256), a 16 KiB tile
// instead of 64 KiB, which held blocks to two per CU; measured for 17 fields at
// 256^3: R2C 0.90 -> 0.85 ms, C2R 1.19 -> 1.13 ms.  FP32: lines_per_block.
template <typename R> __host__ __device__ constexpr int x_lines(int M) {
  return sizeof(R) == 8 ? ((64 / plan_T(M)) > 0 ? 64 / plan_T(M) : 1) : lines_per_block(M);
}
// Of k_x_c2r: the same, and one wave for short lines (FP32, 1 MiB of 24 points: 16.6 us
// with four waves, 15.9 us with one).
__host__ __device__ constexpr bool x_c2r_short(int M, int V) { return plan_T(M, V) <= 2; }
template <typename R> __host__ __device__ constexpr int x_c2r_lines(int M, int V) {
  return (sizeof(R) == 8 || x_c2r_short(M, V)) ? 64 / plan_T(M, V) : lines_per_block(M);
}

constexpr unsigned long kStageBytes = 2ul << 20;

// ---------------------------------------------------------------------------
// Real <-> half-complex x lines on a complex FFT of length M = NX/2.
// z[n] = x[2n] + i x[2n+1];  Z = FFT_M(z);  W = exp(-2 pi i/NX).
//   R2C:  X_k = 1/2 (Z_k + conj Z_{M-k}) - i/2 W^k (Z_k - conj Z_{M-k}),  k = 0..M
//   C2R:  Z_k = (X_k + conj X_{M-k}) + i conj(W^k) (X_k - conj X_{M-k}), k = 0..M-1,
//         with the imaginary parts of X_0 and X_M dropped (Hermitian projection).
// ---------------------------------------------------------------------------
template <typename R>
__device__ __forceinline__ c2<R> r2c_post(c2<R> zk, c2<R> zmk, c2<R> wk, R half_scale) {
  const R ar = zk.x + zmk.x, ai = zk.y - zmk.y;
  const R br = zk.x - zmk.x, bi = zk.y + zmk.y;
  const R cr = wk.x * br - wk.y * bi, ci = wk.x * bi + wk.y * br;
  return mk<R>(half_scale * (ar + ci), half_scale * (ai - cr));
}
template <typename R>
__device__ __forceinline__ c2<R> c2r_pre(c2<R> xk, c2<R> xmk, c2<R> wk) {
  const R ar = xk.x + xmk.x, ai = xk.y - xmk.y;
  const R br = xk.x - xmk.x, bi = xk.y + xmk.y;
  const R cr = wk.x * br + wk.y * bi, ci = wk.x * bi - wk.y * br;
  return mk<R>(ar - ci, ai + cr);
}

// ---------------------------------------------------------------------------
// x pass, forward: real lines (NX) -> half spectrum lines (M main + 1 Nyquist).
// src: real lines; dst: main block (the same memory for an in-place pass: a line
// is read whole, through LDS, before any of it is written); nyq: Nyquist
// entries, one per line.
// tw:  table of exp(-2 pi i q/NX), q in [0, NX).
// ---------------------------------------------------------------------------
template <typename R, int NX>
__global__ void __launch_bounds__(x_lines<R>(NX / 2) * plan_T(NX / 2))
k_x_r2c(const c2<R>* src, c2<R>* dst, c2<R>* __restrict__ nyq, long nlines,
        const c2<R>* __restrict__ tw, R scale) {
  constexpr int M = NX / 2, T = plan_T(M), E = plan_E(M);
  constexpr int LPB = x_lines<R>(M), NT = LPB * T;
  __shared__ c2<R> sh[LPB * M];
  const long l0 = (long)blockIdx.x * LPB;
  const int nl = (int)((nlines - l0) < LPB ? (nlines - l0) : LPB);
  const int l = threadIdx.x / T, t = threadIdx.x % T;
  const bool act = l < nl;
  const c2<R>* gs = src + l0 * M;
  c2<R>* g = dst + l0 * M;
  c2<R> v[E];
  // bank_stays: an in-place pass also finds its input in cache
  const bool keep = bank_stays((unsigned long)nlines * M * sizeof(c2<R>));
  if (keep && src == dst) {
#pragma unroll
    for (int s = 0; s < kInSlots<M>; ++s)
      if (act && rfft_in_valid<M>(t, s)) v[s] = gs[(long)l * M + rfft_in_idx<M>(t, s)];
  } else {
#pragma unroll
    for (int s = 0; s < kInSlots<M>; ++s)
      if (act && rfft_in_valid<M>(t, s)) v[s] = ld_nt<R>(gs + (long)l * M + rfft_in_idx<M>(t, s));
  }
  c2<R>* line = sh + l * M;
  rfft<R, M, false, 1>(v, t, act, line, tw, 2);
  __syncthreads();
#pragma unroll
  for (int s = 0; s < kOutSlots<M>; ++s)
    if (act && rfft_out_valid<M>(t, s)) line[rfft_out_idx<M>(t, s)] = v[s];
  __syncthreads();
  const R hs = R(0.5) * scale;
  for (int i = threadIdx.x; i < nl * M; i += NT) {
    const int ll = i / M, k = i - ll * M;
    const c2<R>* z = sh + ll * M;
    const c2<R> x = r2c_post<R>(z[k], z[(M - k) % M], tw[k], hs);
    if (keep) g[i] = x;
    else st_nt<R>(g + i, x);
  }
  if (threadIdx.x < nl) {
    const c2<R> z0 = sh[threadIdx.x * M];
    nyq[l0 + threadIdx.x] = mk<R>((z0.x - z0.y) * scale, R(0));
  }
}

// ---------------------------------------------------------------------------
// x pass, inverse: half spectrum lines -> real lines (unnormalised); src and dst
// may be the same memory (a block passes a barrier between its reads and its
// writes).  V: plan variant.
// STAGE: short lines, of one or two threads (x_c2r_short), are read and stored through
// LDS: a wave's access from its registers touches 16 or 32 bytes of each of
// 64 or 32 lines, and with the streaming hint those of a cache line go to memory one by
// one.  C2R of a whole transform, 32 x 64 x 48 FP64, 100 MiB: 366 us from registers
// (285 us with no hint), 116 us through LDS.  From four threads on a wave's access fills
// 64 bytes and more (96 x 64 x 48, 99 MiB: 120 us).  Less than kStageBytes goes straight
// from registers, since then the barriers and the way through LDS count (C2R of 24 x 16 x
// 16 FP32, 1.1 MiB: 15.6 us straight and 16.0 staged, 2 MiB alike, 4 MiB 19.3 and 19.1).
// ---------------------------------------------------------------------------
template <typename R, int NX, int V, bool STAGE>
__global__ void __launch_bounds__(x_c2r_lines<R>(NX / 2, V) * plan_T(NX / 2, V))
k_x_c2r(const c2<R>* src, c2<R>* dst, const c2<R>* __restrict__ nyq, long nlines,
        const c2<R>* __restrict__ tw) {
  constexpr int M = NX / 2, T = plan_T(M, V), E = plan_E(M, V);
  constexpr int LPB = x_c2r_lines<R>(M, V), NT = LPB * T;
  constexpr int MP = STAGE ? M + 1 : M;  // row pitch in LDS: a short row's lanes start in other banks
  __shared__ c2<R> sh[(STAGE || plan_np(M, V) > 1) ? LPB * MP : 1];
  const int l = threadIdx.x / T, t = threadIdx.x % T;
  const long l0 = (long)blockIdx.x * LPB, line = l0 + l;
  const int nl = (int)((nlines - l0) < LPB ? (nlines - l0) : LPB);
  const bool act = l < nl;
  const c2<R>* g = src + (act ? line : 0) * M;
  c2<R>* row = sh + ((STAGE || plan_np(M, V) > 1) ? l * MP : 0);
  c2<R> v[E];
  if constexpr (STAGE) {
#pragma unroll
    for (int q = 0; q < M / T; ++q)
      if (const int i = threadIdx.x + q * NT; i < nl * M) v[q] = src[l0 * M + i];
#pragma unroll
    for (int q = 0; q < M / T; ++q)
      if (const int i = threadIdx.x + q * NT; i < nl * M) sh[i / M * MP + i % M] = v[q];
    __syncthreads();
    g = row;
  }
  // pre-processing (X_k and X_{M-k} of the line) straight into registers
#pragma unroll
  for (int s = 0; s < kInSlots<M, V>; ++s) {
    if (!(act && rfft_in_valid<M, V>(t, s))) continue;
    const int k = rfft_in_idx<M, V>(t, s);
    if (k == 0) {
      const R a0 = g[0].x, xn = nyq[line].x;
      v[s] = mk<R>(a0 + xn, a0 - xn);
    } else {
      v[s] = c2r_pre<R>(g[k], g[M - k], tw[k]);
    }
  }
  rfft<R, M, true, 1, V>(v, t, act, row, tw, 2);
  // an in-place pass over a bank that stays in cache (bank_stays) leaves it there
  const bool keep = src == dst && bank_stays((unsigned long)nlines * M * sizeof(c2<R>));
  if constexpr (STAGE) {
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kOutSlots<M, V>; ++s)
      if (rfft_out_valid<M, V>(t, s)) row[rfft_out_idx<M, V>(t, s)] = v[s];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < M / T; ++q)
      if (const int i = threadIdx.x + q * NT; i < nl * M) {
        const c2<R> x = sh[i / M * MP + i % M];
        if (keep) dst[l0 * M + i] = x;
        else st_nt<R>(dst + l0 * M + i, x);
      }
    return;
  }
  c2<R>* gd = dst + (act ? line : 0) * M;
  if (keep) {
#pragma unroll
    for (int s = 0; s < kOutSlots<M, V>; ++s)
      if (act && rfft_out_valid<M, V>(t, s)) gd[rfft_out_idx<M, V>(t, s)] = v[s];
  } else {
#pragma unroll
    for (int s = 0; s < kOutSlots<M, V>; ++s)
      if (act && rfft_out_valid<M, V>(t, s)) st_nt<R>(gd + rfft_out_idx<M, V>(t, s), v[s]);
  }
}

}  // namespace pf
