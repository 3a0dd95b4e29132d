// BitNet W2A8 (int8 x 2-bit) tiled GEMM: the entry point, which picks the translation unit that holds the word
// layout and epilogue asked for (dq_gemm_i2.h).
#include "dq_gemm_i2.h"
#include "dq_gemm_kwaves.h"

namespace dq {

// K over the waves of a workgroup, of row-major words: the form, or -1.  From 17 rows on while the direct-to-LDS kernel's tiles
// are few, from five where K is no multiple of 256, which the register-resident kernel does not take (M = 20, N = 3000, K = 3200
// 17 -> 7.7 us), where the estimate is ahead of that of the kernel that would run.  13 000 shapes of 17 to 600 rows, N 256 to
// 40000, K 256 to 16384: 0.74 of the time without this one in the mean, 0.9 % more than a twentieth slower (M = 39, N = 6544,
// K = 12288 39.7 -> 14.6 us; not M = 27, N = 20384, K = 3840, 10.3 us on the register-resident kernel and 13.2
// here, nor M = 322, N = 4872, K = 256, 6.9 on tiles of 128 x 64 and 10.4).  The three estimates (us):
static constexpr gemm::KwavesCosts kKwavesI2 = {{2.9, 0.9, 0.55, false}, {3.4, 0.80, 0.57, false}, {4.0, 0.73, 0.85, false},
                                                {3.8, 1.84, 1.26, true}, {3.9, 2.21, 1.39, true}};
// the register-resident kernel, whose waves take an eighth of K each in whole pairs of 128-k blocks, beyond K = 8192 in chunks
// of 24 pairs (1947 shapes of 17 to 32 rows, mean error 4.5 %); 0: not its call.  Beyond 32 rows it takes what is at most one and
// a half rounds of workgroups, in chunks one.
static double i2_resident_time(int M, int N, int K) {
  const int pairs = K / 256, chunks = pairs > 32 ? (pairs + 23) / 24 : 1;
  const long wgs = (((long)N + 31) / 32) * (((long)M + 31) / 32);
  if (K % 256 != 0 || M > 128 || (M > 32 && wgs > (chunks > 1 ? 256 : 384))) return 0.0;
  const double steps = 2.048 * chunks * (((pairs + chunks - 1) / chunks + 7) / 8), rounds = (double)((wgs + 255) / 256);
  return 2.0 + 0.84 * steps + rounds * (0.66 + 0.29 * chunks) + 0.36e-3 * K * (double)wgs / 256.0;
}
// the register-staged kernel's tiles of 128 x 64 (3061 shapes of more than 128 rows, K < 4096, mean error 5 %)
static double i2_small_tiles_time(int M, int N, int K) {
  const long tiles = (((long)M + 127) / 128) * (((long)N + 63) / 64);
  const double rounds = (double)((tiles + 255) / 256);
  return 4.75 + 0.91 * rounds + 1e-3 * K * (2.63 * rounds + 0.76 * (double)tiles / 256.0);
}
int i2_kwaves_form(int M, int N, int K) {
  if (M < (K % 256 ? 5 : 17) || half_tiles(M, N) >= gemm::kHalfTileMin) return -1;
  const gemm::KwavesPick pick = gemm::kwaves_pick(kKwavesI2, M, N, K, (size_t)M * K);
  // the K-sliced kernel keeps what its rounds of 256 tiles fill better: M = 200, N = K = 8192 28 us, 29.5 here
  if (K % 2048 == 0 && K >= 4096) {
    const long tiles = (((long)M + 63) / 64) * (((long)N + 127) / 128);
    if (tiles >= 64 && tiles <= 448 && 7.5 + 1.87e-3 * K * (double)((tiles + 255) / 256) < pick.us) return -1;
  }
  // where its waves share K out evenly the estimate is high, the neighbours' as well as it was fitted (M = 117, N = 2592, K = 2048
  // 5.3 us, 6.7 on the register-resident kernel; M = 350, N = 2872 8.9, 11.1 on the tiles): 255 shapes that come here by that take
  // 0.93 of the neighbour's time
  const double even = M <= 1000 ? gemm::kwaves_even(pick, K, 512) : 1.0;
  if (const double resident = i2_resident_time(M, N, K); resident > 0.0)
    return pick.us < 0.96 * resident || even * pick.us < 0.86 * resident ? pick.form : -1;
  // beyond a thousand rows and 8 MiB of activations the estimate of the tiles is high, too (M = 1099, N = 2168, K = 11776 67 us there
  // and 49 here, M = 1900, N = 192, K = 20864 70 and 39, but M = 4037, N = 192, K = 20992 56 and 88)
  const double margin = M > 1000 && (size_t)M * K > (8u << 20) ? 0.78 : 0.94;
  return M <= 64 || even * pick.us < margin * i2_small_tiles_time(M, N, K) ? pick.form : -1;
}

int i2_tile_rows(int M, int N, int K) {
  return gemm::dma_rows<I2Policy<I2_OFFSET, Int32Out<0, false>, true, false, false>>(
      gemm::make_params(nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, M, N, K), kI2HalfTileMin);
}

int i2_gemm(const void* A, const void* B, void* C, int M, int N, int K, int convention, int layout, const void* s_a,
            float s_w, int bitnet_epilogue, int kwaves, hipStream_t stream) {
  gemm::Params p = gemm::make_params(A, B, s_a, nullptr, nullptr, C, M, N, K);
  p.f0 = s_w;
  const bool interleaved = (layout & ~LAYOUT_FRAGMENTS) == LAYOUT_INTERLEAVED;
  if (layout & LAYOUT_FRAGMENTS) return i2_gemm_fragments(p, convention, interleaved, bitnet_epilogue != 0, stream);
  if (interleaved) {
    return bitnet_epilogue ? i2_gemm_interleaved_bitnet(p, convention, kwaves, stream) : i2_gemm_interleaved_int32(p, convention, kwaves, stream);
  }
  return bitnet_epilogue ? i2_gemm_rowmajor_bitnet(p, convention, kwaves, stream) : i2_gemm_rowmajor_int32(p, convention, kwaves, stream);
}

}  // namespace dq
