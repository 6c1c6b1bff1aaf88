// The x-line pass of a batched ensemble group (pf_launch.hpp).
#include "pf_xline_launch.hpp"

namespace pf {
int xline_batch(const StepCall& c, const Member<float>* mt, long nmem, hipStream_t s) {
  return xline_size<float, false, true>(c, nullptr, nullptr, nullptr, nullptr, nmem, false, false, mt, nullptr, s);
}
}  // namespace pf
