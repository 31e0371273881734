// Instantiation of the window kernel for element type bf16_t.
#include "rz_gemm_inst.h"

namespace rz {
hipError_t launch_window_bf16(const WindowParams& p, int windows, hipStream_t stream) {
  return launch_window_t<bf16_t>(p, windows, stream);
}
}  // namespace rz
