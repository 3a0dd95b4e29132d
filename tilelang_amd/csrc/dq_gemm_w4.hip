// uint4 x fp16 on the LDS-staged dequantize GEMM (dq_gemm_core.h): the fine-grained example and W4A16 at large M.
#include "dq_gemm_w4.h"

namespace dq {

using gemm::Params;

// What a call takes on the direct-to-LDS kernel's tiles (us), whichever are best
double w4_tiled_time(int M, int N, int K) {
  using P = W4F16Policy<W4_SCALE, false>;
  const Params p = gemm::make_params(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, M, N, K);
  constexpr int kHeights[4] = {96, 128, 192, 256};
  double best = 1e30;
  for (int i = 0; i < 4; ++i) {
    const double us = P::kRowCosts[i].start + gemm::dma_rounds(gemm::tiles_of(p, kHeights[i])) * (P::kRowCosts[i].round + P::kRowCosts[i].per_k * K * 1e-3);
    if (us < best) best = us;
  }
  return best;
}

int w4_tile_rows(int M, int N, int K, int group, int mode) {
  Params p = gemm::make_params(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, M, N, K);
  p.p0 = (group == K) ? 31 : (31 - __builtin_clz(group));
  return mode >= W4_ZEROS_ORIGINAL ? gemm::dma_rows<W4F16Policy<W4_ZEROS_ORIGINAL, false>>(p)
         : mode >= W4_SCALE        ? gemm::dma_rows<W4F16Policy<W4_SCALE, false>>(p)
                                   : gemm::dma_rows<W4F16Policy<W4_UNSIGNED, false>>(p);
}

int w4_f16_gemm(const void* A, const void* B, const void* S, const void* Z, void* C, int M, int N, int K, int group,
                int mode, int layout, hipStream_t stream) {
  Params p = gemm::make_params(A, B, S, Z, nullptr, C, M, N, K);
  p.p0 = (group == K) ? 31 : (31 - __builtin_clz(group));
  p.p1 = K / group;
#define DQ_W4(MODE_)                                                                                \
  do {                                                                                              \
    if (layout == LAYOUT_PLAIN) return gemm::launch_best<W4F16Policy<MODE_, false>>(p, stream);     \
    return gemm::launch_best<W4F16Policy<MODE_, true>>(p, stream);                                  \
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
