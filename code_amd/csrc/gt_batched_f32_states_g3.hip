// gt_batched_f32_states_g3.hip -- the state variants of the FP32 HALFSPLIT
// strip kernels (gt_strip_impl.h) with 3 tracers per wavefront.
#include "gt_strip_impl.h"

namespace gt {

hipError_t launch_states_f32_g6(hipStream_t st, const FusedArgs<float>& a);
hipError_t launch_states_f32(hipStream_t st, const FusedArgs<float>& a, int group) {
  return group == 6 ? launch_states_f32_g6(st, a) : dispatch_states<float, 3, false>(st, a);
}

}  // namespace gt
