// The x-line passes in FP32 (pf_launch.hpp).
#include "pf_xline_launch.hpp"

namespace pf {
template int xline<float>(bool, const StepCall&, c2<float>*, c2<float>*, float*, double*, long*, bool, bool, hipStream_t);
template bool xline_accepts<float>(const Geo&, int);
}  // namespace pf
