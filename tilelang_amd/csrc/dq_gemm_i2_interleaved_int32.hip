// BitNet W2A8 (int8 x 2-bit) tiled GEMM: the kernels for interleaved words and the int32 epilogue (dq_gemm_i2.h).
#include "dq_gemm_i2.h"

namespace dq {

int i2_gemm_interleaved_int32(const gemm::Params& p, int convention, int kwaves, hipStream_t stream) {
  return i2_gemm_part<true, false, false>(p, convention, kwaves, stream);
}

}  // namespace dq
