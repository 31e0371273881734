// Instantiation of the backward pass in one launch for element type bf16_t.
#include "rz_gemm_inst.h"

namespace rz {
hipError_t launch_backward_bf16(GemmParams ig, const SplitPlan* split, GemmParams wg, const WeightGradPlan* plan, const BackwardForm& form,
                        hipStream_t stream) {
  return launch_backward_t<bf16_t>(ig, split, wg, plan, form, stream);
}
hipError_t launch_input_grad_pack_bf16(const GemmParams& ig, const SplitPlan* split, const WindowParams& w, const PackForm& form,
                                       hipStream_t stream) {
  return launch_input_grad_pack_t<bf16_t>(ig, split, w, form, stream);
}
}  // namespace rz
