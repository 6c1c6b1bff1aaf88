// Launchers of the FP64 faithful step's kernels (pf_faithful.hip).
#pragma once
#include "pf_step_kernels.hpp"

namespace pf {

constexpr int kNlBlock = 256;

// Loops 5-10 of the real state bank st (c, eta_1..) into the bank dfd (df_dc,
// df_dphi_1..) and mobd = mob_c - D_mean; with diag six block partials (f_ch,
// f_eta, c_max, c_min, phi_min, phi_3) per block in part.
int faithful_nonlinear(const Geo& g, const UPar& u, bool diag, const double* st, double* dfd, double* mobd,
                       double* part, long max_blocks, long* nblocks, hipStream_t s);

// One k-space pass over the z columns of fields f0 .. f0+nf-1 (k_zfaithful):
// U the state bank, D the derivatives', G the mobility chain's one field.  With
// pars one block partial of f_int per block in part.
enum { FZ_ETA = 0, FZ_GHAT = 1, FZ_CMOB = 2 };
int faithful_z(int role, bool pars, const Geo& g, const UPar& u, const KTab& kt, Bank<double> U, Bank<double> D,
               Bank<double> G, double* part, int f0, int nf, long max_blocks, long* nblocks, hipStream_t s);

}  // namespace pf
