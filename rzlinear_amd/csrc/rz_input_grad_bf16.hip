// Instantiation of the input-grad contraction kernels for element type bf16_t.
#include "rz_gemm_inst.h"

namespace rz {
hipError_t launch_input_grad_bf16(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning,
                        hipStream_t stream) {
  return launch_gemm_t<bf16_t, kInputGrad>(p, plan, split, tuning, stream);
}
}  // namespace rz
