// gt_batched_f64_g2.hip -- FP64 (reference-exact) instantiations of the
// HALFSPLIT strip kernels (gt_strip_impl.h): two tracers per wavefront.
#include "gt_strip_impl.h"

namespace gt {

hipError_t launch_fused_f64_g2(hipStream_t st, const FusedArgs<double>& a) {
  return dispatch_scheme<double, 2, true, false>(st, a);
}

}  // namespace gt
