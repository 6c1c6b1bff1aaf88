// The z-line pass of a batched ensemble group (pf_launch.hpp).
#include "pf_zline_launch.hpp"

namespace pf {
int zline_batch(const StepCall& c, const Member<float>* mt, long nmem, hipStream_t s) {
  const Bank<float> none{nullptr, nullptr};
  return zline_size<float, ROLE_REG, true, false, true>(c, none, none, none, none, nullptr, nullptr, 0,
                                                        (int)(nmem * c.g.F), mt, nullptr, s);
}
}  // namespace pf
