// The y and z passes of the 3-D transform over a bank in the split-Nyquist
// layout (pf_kernels.hpp), each one launch over the main block and the Nyquist
// planes together.  Both are bound by HBM (or, for banks that fit it, by the last
// level cache): 5.3 TB/s for one FP64 field of 256^3, 5.6 TB/s for 17.  A whole
// R2C with its C2R, caller's layout to caller's layout, moves 12 times the data
// instead of 20: 0.65 -> 0.33 ms for one FP64 256^3 field (kz fastest), 0.48 ->
// 0.30 ms for 9 FP32 fields of 192 x 160 x 96 (kx fastest).
#pragma once
#include "pf_kernels.hpp"
#include "pf_step_kernels.hpp"

namespace pf {

// ---------------------------------------------------------------------------
// k_ypass: y transform of np panels (z, field) of the main block and of as many
// contiguous lines of the Nyquist planes.  Both are the same work with other
// strides, so one code path serves them: a tile is TX transforms ("columns"),
// element e of column c at c * (column stride) + e * (element stride),
//   main block    : columns kx, NY rows of M elements a panel; the columns of all
//                   panels are numbered through, so tiles of a row shorter than
//                   TX, or no multiple of it, carry no padding columns
//   Nyquist planes: columns are the lines, NY contiguous elements each.
// A wave's lanes run along whichever of the two is contiguous.  The Nyquist tiles,
// whose LDS exchanges run against the lanes, come first, so that they end under the
// rest (ypass_grid blocks).
// BATCH: the W banks of every member in mt, ppm panels (and Nyquist lines) per
// member; main and nyq are unused.
// ---------------------------------------------------------------------------
// The grid: an eighth of each kind's tiles (rounded up) per XCD.
inline unsigned ypass_grid(long tmain, long tnyq) { return (unsigned)(8 * ((tmain + 7) / 8 + (tnyq + 7) / 8)); }

// Whether a Nyquist tile exchanges each line in LDS elements of its own rather than in
// the tile's column order, where the lanes of a line, TX elements apart, share a bank.
// With more than one exchange, or 16 threads a line and 8-byte elements, the few
// Nyquist tiles of a small bank otherwise outlast the rest: a y pass of 24 x 512 x 24 x
// 6 FP32 20.4 us in column order, 11.6 us in rows; 24 x 192 x 24 x 6 11.3 and 7.7, FP64
// 10.3 and 8.9; 24 x 256 x 24 x 6 FP32 9.9 and 8.2.  Elsewhere it gains nothing, and the
// second copy of the transform costs the main block's tiles a little (128 x 256 x 64 x 9
// FP64 48.2 and 49.3 us; where it is used, 128 x 512 x 64 x 9 FP32 52.8 and 53.9).
template <typename R> __host__ __device__ constexpr bool ypass_own_rows(int NY) {
  return plan_np(NY) > 2 || (plan_np(NY) == 2 && plan_T(NY) >= 16 && sizeof(R) == 4);
}

// KEEP: the bank stays in cache from pass to pass (bank_stays).
template <typename R, int NY, bool INV, bool BATCH = false, bool KEEP = false>
__global__ void __launch_bounds__(col_tile(NY, sizeof(c2<R>)) * plan_T(NY))
k_ypass(c2<R>* __restrict__ main, c2<R>* __restrict__ nyq, long M, long npanels, long nlines,
        const c2<R>* __restrict__ tw, const Member<R>* __restrict__ mt, long ppm) {
  constexpr int E = plan_E(NY), T = plan_T(NY);
  constexpr unsigned TX = col_tile(NY, sizeof(c2<R>)), CB = sizeof(c2<R>);
  static_assert(last_pass_in_place<NY>(), "slot rows of the last pass are t + a per-slot constant");
  __shared__ c2<R> sh[(plan_np(NY) > 1) ? NY * TX : 1];
  const unsigned m = (unsigned)M, np = (unsigned)(BATCH ? ppm : npanels), nl = (unsigned)(BATCH ? ppm : nlines);
  const unsigned nmem = BATCH ? (unsigned)(npanels / ppm) : 1u;
  const unsigned tmain = (np * m + TX - 1) / TX, tnyq = (nl + TX - 1) / TX;  // tiles per member
  // XCD x (blocks x, x + 8, ...) takes every eighth Nyquist tile, then one
  // contiguous range of main-block tiles (their 128-byte pieces of the same rows
  // are read by one XCD at about the same time).
  const unsigned x = blockIdx.x % 8, i = blockIdx.x / 8, nq = (tnyq * nmem + 7) / 8;
  const bool isn = i < nq;
  unsigned b = isn ? i * 8 + x : x * (gridDim.x / 8 - nq) + (i - nq);
  c2<R>* base = isn ? nyq : main;
  if constexpr (BATCH) {
    const unsigned mem = b / (isn ? tnyq : tmain);
    if (mem >= nmem) return;  // one of the grid's rounding blocks
    b -= mem * (isn ? tnyq : tmain);
    base = isn ? mt[mem].Wn : mt[mem].Wm;
  }
  const unsigned c = isn ? threadIdx.x / T : threadIdx.x % TX, t = isn ? threadIdx.x % T : threadIdx.x / TX;
  bool act;
  unsigned voff, es;  // lane byte offset, byte stride of the rows
  unsigned long left;  // bytes of the bank from base on
  if (!isn) {
    const unsigned q0 = b * TX, p0 = q0 / m, r = q0 - p0 * m + c;
    act = q0 + c < np * m;
    const unsigned dp = (q0 - p0 * m + TX <= m) ? 0u : r / m;  // panels past the tile's first
    base += (unsigned long)p0 * NY * m;
    left = p0 < np ? (unsigned long)(np - p0) * NY * m * CB : 0ul;
    es = m * CB;
    voff = (dp * ((unsigned)NY - 1u) * m + r) * CB + t * es;
  } else {
    const unsigned l0 = b * TX;
    act = l0 + c < nl;
    base += (unsigned long)l0 * NY;
    left = (unsigned long)TX * NY * CB;
    es = CB;
    voff = (c * NY + t) * CB;
  }
  // a bank that stays in cache: plain accesses through a buffer descriptor, lanes
  // without a column out of its range; a streamed one: hinted accesses by pointer
  // (256^3 x 17 FP32: 428 us by pointer, 438 us through the descriptor)
  const BufRes rb = buf_res(base, left < 0xFFFFFFF0ul ? (unsigned)left : 0xFFFFFFF0u);
  c2<R>* const gp = reinterpret_cast<c2<R>*>(reinterpret_cast<char*>(base) + voff);
  const unsigned ee = es / CB;
  c2<R> v[E];
  if constexpr (KEEP) {
    if (!act) voff = kBufOut;
#pragma unroll
    for (int s = 0; s < kInSlots<NY>; ++s)
      if (rfft_in_valid<NY>(t, s)) v[s] = buf_ld<R, 0>(rb, voff, (unsigned)rfft_in_idx<NY>(0, s) * es);
  } else {
#pragma unroll
    for (int s = 0; s < kInSlots<NY>; ++s)
      if (act && rfft_in_valid<NY>(t, s)) v[s] = ld_nt<R>(gp + (unsigned long)rfft_in_idx<NY>(0, s) * ee);
  }
  if (ypass_own_rows<R>(NY) && isn) rfft<R, NY, INV, 1>(v, t, KEEP || act, sh + c * NY, tw);
  else rfft<R, NY, INV, (int)TX>(v, t, KEEP || act, sh + c, tw);
  if constexpr (KEEP) {
#pragma unroll
    for (int s = 0; s < kOutSlots<NY>; ++s)
      if (rfft_out_valid<NY>(t, s)) buf_st<R, 0>(rb, voff, (unsigned)rfft_out_idx<NY>(0, s) * es, v[s]);
  } else {
#pragma unroll
    for (int s = 0; s < kOutSlots<NY>; ++s)
      if (act && rfft_out_valid<NY>(t, s)) st_nt<R>(gp + (unsigned long)rfft_out_idx<NY>(0, s) * ee, v[s]);
  }
}

// ---------------------------------------------------------------------------
// k_zpass: z transform of nf fields between the split layout (near side) and the
// layout FAR: forward reads near and writes far, inverse reads far and writes
// near.  So the last forward pass delivers the caller's layout (and the first
// inverse one takes it) with no repacking pass.
//   FAR_SPLIT: the split layout at far, farn (may be near itself)
//   FAR_TILED: the column-tile layout of the carried spectrum (Geo), at far
//   FAR_XFAST: dense (nz, ny, M+1), kx fastest, at far
//   FAR_ZFAST: dense (M+1, ny, nz), kz fastest, at far
// One tile of TX columns per block: tiles 0 .. tm-1 of a field over its M*ny
// main-block columns, tn more over the ny Nyquist-plane columns.
// ---------------------------------------------------------------------------
enum { FAR_XFAST = 0, FAR_ZFAST = 1, FAR_SPLIT = 2, FAR_TILED = 3 };

template <typename R, int NZ, bool INV, int FAR>
__global__ void __launch_bounds__(col_tile(NZ, sizeof(c2<R>)) * plan_T(NZ))
k_zpass(c2<R>* near, c2<R>* nearn, c2<R>* far, c2<R>* farn, unsigned M, unsigned ny, unsigned nf, unsigned tm,
        unsigned tn, unsigned run_tiles, const c2<R>* __restrict__ tw) {
  constexpr int E = plan_E(NZ);
  constexpr unsigned TX = col_tile(NZ, sizeof(c2<R>)), CB = sizeof(c2<R>);
  static_assert(last_pass_in_place<NZ>(), "slot rows of the last pass are t + a per-slot constant");
  __shared__ c2<R> sh[(plan_np(NZ) > 1) ? NZ * TX : 1];
  const unsigned tpf = tm + tn;
  const unsigned tile = (unsigned)xcd_runs(blockIdx.x, gridDim.x, run_tiles);
  const unsigned f = tile / tpf, tt = tile - f * tpf;
  if (f >= nf) return;  // the grid is rounded up to whole XCD runs
  const bool isn = tt >= tm;
  const unsigned W = isn ? ny : M * ny, col0 = (isn ? tt - tm : tt) * TX;
  const unsigned c = threadIdx.x % TX, t = threadIdx.x / TX;
  const bool act = col0 + c < W;
  const unsigned long fmain = (unsigned long)f * M * ny * NZ, fplane = (unsigned long)f * ny * NZ;
  const unsigned nrow = W * CB;
  const BufRes rn = buf_res((isn ? nearn + fplane : near + fmain) + col0, (unsigned)NZ * nrow);
  const unsigned noff = act ? (t * W + c) * CB : kBufOut;
  unsigned foff, frow;
  BufRes rf = rn;
  if constexpr (FAR == FAR_SPLIT) {
    rf = buf_res((isn ? farn + fplane : far + fmain) + col0, (unsigned)NZ * nrow);
    frow = nrow;
    foff = noff;
  } else if constexpr (FAR == FAR_TILED) {
    rf = buf_res(far + ((unsigned long)f * tpf + tt) * (NZ * TX), NZ * TX * CB);
    frow = TX * CB;
    foff = act ? threadIdx.x * CB : kBufOut;
  } else {
    const unsigned long half = fmain + fplane;
    const unsigned col = act ? col0 + c : 0u;
    const unsigned ky = isn ? col : col / M, kx = isn ? M : col - ky * M;
    rf = buf_res(far + half, (M + 1) * ny * NZ * CB);
    frow = (FAR == FAR_XFAST ? ny * (M + 1) : 1u) * CB;
    foff = act ? (FAR == FAR_XFAST ? ky * (M + 1) + kx : (kx * ny + ky) * NZ) * CB + t * frow : kBufOut;
  }
  // near: the scratch bank (or the bank itself), by bank_stays; far: dense layouts
  // have rows of no whole cache lines, neighbouring tiles (XFAST) or slots (ZFAST)
  // share lines and the accesses keep them in L2; the carried spectrum's tiles are
  // streamed
  const bool keep = bank_stays((unsigned long)nf * M * ny * NZ * CB);
  constexpr int AUXF = (FAR == FAR_XFAST || FAR == FAR_ZFAST) ? 0 : kBufNT;
  constexpr bool NEARIN = !INV, NEAROUT = INV || FAR == FAR_SPLIT;
  c2<R> v[E];
  if (NEARIN && keep) {
#pragma unroll
    for (int s = 0; s < kInSlots<NZ>; ++s)
      if (rfft_in_valid<NZ>(t, s)) v[s] = buf_ld<R, 0>(rn, noff, (unsigned)rfft_in_idx<NZ>(0, s) * nrow);
  } else {
#pragma unroll
    for (int s = 0; s < kInSlots<NZ>; ++s)
      if (rfft_in_valid<NZ>(t, s)) {
        const unsigned i = (unsigned)rfft_in_idx<NZ>(0, s);
        v[s] = NEARIN ? buf_ld<R>(rn, noff, i * nrow) : buf_ld<R, AUXF>(rf, foff, i * frow);
      }
  }
  rfft<R, NZ, INV, (int)TX>(v, t, true, sh + c, tw);
  if (NEAROUT && keep) {
#pragma unroll
    for (int s = 0; s < kOutSlots<NZ>; ++s)
      if (rfft_out_valid<NZ>(t, s))
        buf_st<R, 0>(INV ? rn : rf, INV ? noff : foff, (unsigned)rfft_out_idx<NZ>(0, s) * (INV ? nrow : frow), v[s]);
  } else {
#pragma unroll
    for (int s = 0; s < kOutSlots<NZ>; ++s)
      if (rfft_out_valid<NZ>(t, s)) {
        const unsigned i = (unsigned)rfft_out_idx<NZ>(0, s);
        if (INV) buf_st<R>(rn, noff, i * nrow, v[s]);
        else buf_st<R, AUXF>(rf, foff, i * frow, v[s]);
      }
  }
}

}  // namespace pf
