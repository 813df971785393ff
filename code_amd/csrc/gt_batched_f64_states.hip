// gt_batched_f64_states.hip -- the state variants of the FP64 HALFSPLIT strip
// kernels (gt_strip_impl.h).
#include "gt_strip_impl.h"

namespace gt {

hipError_t launch_states_f64(hipStream_t st, const FusedArgs<double>& a) {
  return dispatch_states<double, 1, true>(st, a);
}

}  // namespace gt
