// Instantiation of the window kernel for element type float.
#include "rz_gemm_inst.h"

namespace rz {
hipError_t launch_window_f32(const WindowParams& p, int windows, hipStream_t stream) {
  return launch_window_t<float>(p, windows, stream);
}
}  // namespace rz
