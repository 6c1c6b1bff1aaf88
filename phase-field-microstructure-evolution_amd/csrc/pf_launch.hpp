// Launches of the fused step kernels (k_xline, k_zline of pf_fused.hpp): size, role
// and policy dispatch.  The instantiations are spread over pf_xline_*.hip and
// pf_zline_*.hip (FP32, FP64 and the batched ensemble's), which define them from
// pf_xline_launch.hpp and pf_zline_launch.hpp.
#pragma once
#include "../../include/pf.h"
#include "pf_fused.hpp"
#include "pf_internal.hpp"

namespace pf {

// The z-line kernel streams four banks with short (TX-column) row segments;
// more resident tiles per CU keep more rows in flight (measured 2.5% faster
// at 32768 than at 8192 blocks, 256^3 x 17 fields).
constexpr long kZlineMaxGrid = 32768;

// Blocks of an x-line pass that leaves diagnostics, and of the pointwise kernels.
constexpr long kMaxGrid = 8192;

struct StepCall {
  const Geo& g;
  const UPar& u;
  const KTab& kt;
  const pf_tuning& tune;
};

// One pass over fields f0 .. f0+nf-1 (role: ROLE_*); with parseval one block
// partial of the next step's f_int per block in part.
template <typename R>
int zline(int role, bool parseval, const StepCall& c, Bank<R> S, Bank<R> W, Bank<R> X, Bank<R> Y, double* dc64,
          double* part, int f0, int nf, long* nblocks, hipStream_t s);
// ROLE_REG of every field of nmem members (FP32, no diagnostics).
int zline_batch(const StepCall& c, const Member<float>* mt, long nmem, hipStream_t s);


// The x-line pass of every field, or (xonly) of the mobility chain's one field;
// with diag six block partials per block in part.
template <typename R>
int xline(bool xonly, const StepCall& c, c2<R>* wm, c2<R>* wn, R* mobd, double* part, long* nblocks, bool diag,
          bool mob, hipStream_t s);
// The faithful step's x pass (k_xline's FAITH) on the bank U of 2F fields, whose state
// is real or x-half lines; var <= kNlRegs.
int xline_faithful(const StepCall& c, bool real, Bank<double> U, double* mobd, double* part, long* nblocks,
                   bool diag, hipStream_t s);
// Whether the x-line takes this grid and field count in blocks of `lines` lines (0:
// of some number).
template <typename R> bool xline_accepts(const Geo& g, int lines);
// The x-line pass of nmem members (FP32, no diagnostics).
int xline_batch(const StepCall& c, const Member<float>* mt, long nmem, hipStream_t s);

}  // namespace pf
