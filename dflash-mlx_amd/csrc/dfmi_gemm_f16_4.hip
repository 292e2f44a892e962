// qmm_gemm_kernel for f16 activations and 4-bit weights.
#include "dfmi_gemm.h"

namespace dfmi {
void gemm_launch_f16_4(int cfg, int gs, const GemmArgs& a, hipStream_t st) {
  gemm_launch_bits<F16, 4>(cfg, gs, a, st);
}
}  // namespace dfmi
