// The x-line passes in FP64 (pf_launch.hpp).
#include "pf_xline_launch.hpp"

namespace pf {
template int xline<double>(bool, const StepCall&, c2<double>*, c2<double>*, double*, double*, long*, bool, bool, hipStream_t);
template bool xline_accepts<double>(const Geo&, int);
}  // namespace pf
