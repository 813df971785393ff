// gt_batched_f64_adv.hip -- FP64 (reference-exact) instantiations of the
// HALFSPLIT strip kernels (gt_strip_impl.h): one tracer and its advective term.
#include "gt_strip_impl.h"

namespace gt {

hipError_t launch_fused_f64_adv(hipStream_t st, const FusedArgs<double>& a) {
  return dispatch_scheme<double, 1, true, true>(st, a);
}

hipError_t launch_strip_uv_adv(hipStream_t st, const FusedArgs<double>& a) {
  return launch_uv<double, 1, true>(st, a);
}

}  // namespace gt
