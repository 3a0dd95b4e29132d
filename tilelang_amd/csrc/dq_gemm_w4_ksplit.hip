// uint4 x fp16 with K cut over workgroups (dq_gemm_core.h): W4A16 at more rows than the streaming kernel is good for, against a
// matrix of few tiles.  The scaled modes.
#include "dq_gemm_w4.h"

namespace dq {

// K in `split` slices with fp32 sums in parts[split][M][N]; 1: not a shape (or a mode) of that kernel
int w4_f16_gemm_ksplit(const void* A, const void* B, const void* S, const void* Z, void* C, void* parts, int M, int N, int K,
                       int group, int mode, int layout, int split, hipStream_t stream) {
  Params p = gemm::make_params(A, B, S, Z, nullptr, C, M, N, K);
  p.p0 = (group == K) ? 31 : (31 - __builtin_clz(group));
  p.p1 = K / group;
  if (group == K) return 1;
#define DQ_W4(MODE_)                                                                                              \
  do {                                                                                                            \
    if (layout == LAYOUT_PLAIN) return gemm::launch_ksplit<W4F16Policy<MODE_, false>>(p, parts, split, stream);   \
    return gemm::launch_ksplit<W4F16Policy<MODE_, true>>(p, parts, split, stream);                                \
  } while (0)
  switch (mode) {
    case W4_SCALE: DQ_W4(W4_SCALE);
    case W4_USCALE: DQ_W4(W4_USCALE);
    case W4_ZEROS_ORIGINAL: DQ_W4(W4_ZEROS_ORIGINAL);
    case W4_ZEROS_FOLDED: DQ_W4(W4_ZEROS_FOLDED);
    default: return 1;
  }
#undef DQ_W4
}

}  // namespace dq
