// Instantiation of the weight-grad contraction kernels for element type float.
#include "rz_gemm_inst.h"

namespace rz {
hipError_t launch_weight_grad_f32(GemmParams p, const WeightGradPlan* plan, const SplitPlan* split, const rz_tuning& tuning,
                        hipStream_t stream) {
  return launch_gemm_t<float, kWeightGrad>(p, plan, split, tuning, stream);
}
}  // namespace rz
