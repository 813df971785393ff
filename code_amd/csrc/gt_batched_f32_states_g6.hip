// gt_batched_f32_states_g6.hip -- the state variants of the FP32 HALFSPLIT
// strip kernels (gt_strip_impl.h) with 6 tracers per wavefront.
#include "gt_strip_impl.h"

namespace gt {

hipError_t launch_states_f32_g6(hipStream_t st, const FusedArgs<float>& a) {
  return dispatch_states<float, 6, false>(st, a);
}

}  // namespace gt
