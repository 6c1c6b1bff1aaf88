// The z-line passes in FP64 (pf_launch.hpp).
#include "pf_zline_launch.hpp"

namespace pf {
template int zline<double>(int, bool, const StepCall&, Bank<double>, Bank<double>, Bank<double>, Bank<double>, double*, double*, int, int,
                          long*, hipStream_t);
}  // namespace pf
