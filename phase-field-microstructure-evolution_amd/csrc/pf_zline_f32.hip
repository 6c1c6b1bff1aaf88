// The z-line passes in FP32 (pf_launch.hpp).
#include "pf_zline_launch.hpp"

namespace pf {
template int zline<float>(int, bool, const StepCall&, Bank<float>, Bank<float>, Bank<float>, Bank<float>, double*, double*, int, int,
                          long*, hipStream_t);
}  // namespace pf
