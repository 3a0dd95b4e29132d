// BitNet W2A8 (int8 x 2-bit) tiled GEMM: the entry point, which picks the translation unit that holds the word
// layout and epilogue asked for (dq_gemm_i2.h).
#include "dq_gemm_i2.h"
#include "dq_gemm_kwaves.h"

namespace dq {

// K over the waves of a workgroup, of row-major words: the form, or -1.  From 17 rows on while the direct-to-LDS kernel's tiles
// are few, against the register-resident, K-sliced and register-staged kernels (230 shapes of 17 to 500 rows; with the layer's
// quantiser M = 20, N = 17328, K = 2560 13.1 -> 11.8 us, M = 37, N = 7216, K = 12288 38 -> 17, M = 145, N = 8296, K = 2048
// 24 -> 12.7, M = 275, N = 2280, K = 10240 30 -> 22; M = 88, N = 2296, K = 2048 7.2 -> 7.5), from five where K is no multiple of
// 256, which the register-resident kernel does not take (M = 20, N = 3000, K = 3200 17 -> 7.7).  The K-sliced kernel keeps what
// its rounds of 256 tiles fill better: M = 200, N = K = 8192 28 us, 29.5 here.
static constexpr gemm::KwavesCosts kKwavesI2 = {{2.9, 0.9, 0.55, false}, {3.4, 0.80, 0.57, false}, {4.0, 0.73, 0.85, false},
                                                {3.8, 1.84, 1.26, true}, {3.9, 2.21, 1.39, true}};
int i2_kwaves_form(int M, int N, int K) {
  if (M < (K % 256 ? 5 : 17) || gemm::kwaves_big_tiles(M, N) >= gemm::kHalfTileMin) return -1;
  const gemm::KwavesPick pick = gemm::kwaves_pick(kKwavesI2, M, N, K);
  if (K % 2048 == 0 && K >= 4096) {
    const long tiles = (((long)M + 63) / 64) * (((long)N + 127) / 128);  // of the K-sliced kernel
    if (tiles >= 64 && tiles <= 448 && 7.5 + 1.87e-3 * K * (double)((tiles + 255) / 256) < pick.us) return -1;
  }
  return pick.form;
}

int i2_gemm(const void* A, const void* B, void* C, int M, int N, int K, int convention, int layout, const void* s_a,
            float s_w, int bitnet_epilogue, int kwaves, hipStream_t stream) {
  gemm::Params p = gemm::make_params(A, B, s_a, nullptr, nullptr, C, M, N, K);
  p.f0 = s_w;
  p.kwaves = kwaves;
  const bool interleaved = (layout & ~LAYOUT_FRAGMENTS) == LAYOUT_INTERLEAVED;
  if (layout & LAYOUT_FRAGMENTS) return i2_gemm_fragments(p, convention, interleaved, bitnet_epilogue != 0, stream);
  if (interleaved) {
    return bitnet_epilogue ? i2_gemm_interleaved_bitnet(p, convention, stream) : i2_gemm_interleaved_int32(p, convention, stream);
  }
  return bitnet_epilogue ? i2_gemm_rowmajor_bitnet(p, convention, stream) : i2_gemm_rowmajor_int32(p, convention, stream);
}

}  // namespace dq
