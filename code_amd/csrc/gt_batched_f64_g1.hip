// gt_batched_f64_g1.hip -- FP64 (reference-exact) instantiations of the
// HALFSPLIT strip kernels (gt_strip_impl.h): one tracer per wavefront.
#include "gt_strip_impl.h"

namespace gt {

hipError_t launch_fused_f64_g1(hipStream_t st, const FusedArgs<double>& a) {
  return dispatch_scheme<double, 1, true, false>(st, a);
}

hipError_t launch_strip_uv_g1(hipStream_t st, const FusedArgs<double>& a) {
  return launch_uv<double, 1, false>(st, a);
}

}  // namespace gt
