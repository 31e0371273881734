// Instantiation of the backward pass in one launch for element type float.
#include "rz_gemm_inst.h"

namespace rz {
hipError_t launch_backward_f32(GemmParams ig, const SplitPlan* split, GemmParams wg, const WeightGradPlan* plan, const BackwardForm& form,
                        hipStream_t stream) {
  return launch_backward_t<float>(ig, split, wg, plan, form, stream);
}
}  // namespace rz
