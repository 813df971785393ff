// gt_batched_f64_mom.hip -- the momentum variants of the FP64 HALFSPLIT strip
// kernels (gt_strip_impl.h).
#include "gt_strip_impl.h"

namespace gt {

hipError_t launch_momentum_f64(hipStream_t st, const FusedArgs<double>& a, int part) {
#define GT_M(S) \
  return part == 0 ? launch_momentum_one<S, MOM_U>(st, a) : launch_momentum_one<S, MOM_V>(st, a)
  switch (a.hscheme) {
    case P2_PDM: GT_M(P2_PDM);
    case SUPERBEE: GT_M(SUPERBEE);
    case MUSCL: GT_M(MUSCL);
    case P2: GT_M(P2);
    case UPSTREAM: GT_M(UPSTREAM);
    default: return hipErrorInvalidValue;
  }
#undef GT_M
}

}  // namespace gt
