// qmm_gemm_kernel for f16 activations and 8-bit weights.
#include "dfmi_gemm.h"

namespace dfmi {
void gemm_launch_f16_8(int cfg, int gs, const GemmArgs& a, hipStream_t st) {
  gemm_launch_bits<F16, 8>(cfg, gs, a, st);
}
}  // namespace dfmi
