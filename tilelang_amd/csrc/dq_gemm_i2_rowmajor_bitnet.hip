// BitNet W2A8 (int8 x 2-bit) tiled GEMM: the kernels for row-major words and the BitLinear fp16 epilogue (dq_gemm_i2.h).
#include "dq_gemm_i2.h"

namespace dq {

int i2_gemm_rowmajor_bitnet(const gemm::Params& p, int convention, int kwaves, hipStream_t stream) {
  return i2_gemm_part<false, true, false>(p, convention, kwaves, stream);
}

}  // namespace dq
