// uint4 x fp16 with K over the waves of a workgroup (dq_gemm_kwaves.h): W4A16 at 3 to some hundreds of rows, where the decode
// kernels do not take the shape or are behind.
#include "dq_gemm_kwaves.h"
#include "dq_gemm_w4.h"

namespace dq {

static constexpr gemm::KwavesCosts kKwavesW4 = {{2.55, 0.92, 1.16, true}, {2.68, 0.97, 1.31, true}, {1.93, 1.92, 2.28, true},
                                                {2.81, 2.41, 2.84, true}, {3.68, 1.91, 3.1, true}};

double w4_kwaves_time(int M, int N, int K) { return gemm::kwaves_pick(kKwavesW4, M, N, K).us; }
int w4_kwaves_form(int M, int N, int K) { return gemm::kwaves_pick(kKwavesW4, M, N, K).form; }

// form: of kKwavesForms, -1 the best by the times.  1: not a shape of that kernel
int w4_f16_gemm_kwaves(const void* A, const void* B, const void* S, const void* Z, void* C, int M, int N, int K, int group,
                       int mode, int layout, int form, hipStream_t stream) {
  Params p = gemm::make_params(A, B, S, Z, nullptr, C, M, N, K);
  p.p0 = (group == K) ? 31 : (31 - __builtin_clz(group));
  p.p1 = K / group;
  if (form < 0) form = w4_kwaves_form(M, N, K);
#define DQ_W4(MODE_)                                                                                         \
  do {                                                                                                       \
    if (!gemm::kwaves_takes<W4F16Policy<MODE_, false>>(p)) return 1;                                         \
    if (layout == LAYOUT_PLAIN) return gemm::launch_kwaves<W4F16Policy<MODE_, false>>(p, form, stream);      \
    return gemm::launch_kwaves<W4F16Policy<MODE_, true>>(p, form, stream);                                   \
  } while (0)
  switch (mode) {
    case W4_UNSIGNED: DQ_W4(W4_UNSIGNED);
    case W4_SIGNED: DQ_W4(W4_SIGNED);
    case W4_OFFSET8: DQ_W4(W4_OFFSET8);
    case W4_SCALE: DQ_W4(W4_SCALE);
    case W4_USCALE: DQ_W4(W4_USCALE);
    case W4_ZEROS_ORIGINAL: DQ_W4(W4_ZEROS_ORIGINAL);
    case W4_ZEROS_RESCALE: DQ_W4(W4_ZEROS_RESCALE);
    case W4_ZEROS_FOLDED: DQ_W4(W4_ZEROS_FOLDED);
    default: DQ_FAIL("w4 fp16 gemm: unknown mode %d", mode);
  }
#undef DQ_W4
}

}  // namespace dq
