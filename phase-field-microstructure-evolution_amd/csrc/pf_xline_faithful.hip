// The faithful step's x pass (pf_launch.hpp).
#include "pf_xline_launch.hpp"

namespace pf {
int xline_faithful(const StepCall& c, bool real, Bank<double> U, double* mobd, double* part, long* nblocks,
                   bool diag, hipStream_t s) {
  switch (c.g.nx) {
#define PF_CASE(N) \
  case N: return xline_faithful_of<N>(c, real, U, mobd, part, nblocks, diag, s);
    PF_GRID_SIZES(PF_CASE)
#undef PF_CASE
    default: return fail(PF_EINVAL, "unsupported nx");
  }
}
}  // namespace pf
