// Shared skeleton of the LDS-staged dequantize-GEMM kernels for gfx950.
//
// Replaces the T.Pipelined / T.copy / T.gemm loop the reference's examples share
// (e.g. examples/dequantize_gemm/example_dequant_gemm_bf16_mxfp4_cdna4.py:231-244,
// example_dequant_gemm_w4a8.py:132-147, examples/bitnet-1.58b/kernel_benchmark/
// tilelang_bitnet_158_int8xint2_prefill.py:238-296) and the tl::gemm_ss template it lowers to
// (src/tl_templates/hip/gemm.h:158-232).  One kernel template, instantiated per weight format
// through a policy:
//
//   * block tile 256 x 256 x BK (BK = 128 bytes of A per row: 64 x 16-bit or 128 x int8), 4 waves
//     as 2 x 2, 128 x 128 per wave = 4 x 4 MFMA 32x32 accumulators (256 registers per lane);
//   * A (transformed by the policy, 16 bytes at a time, on its way through registers) and the
//     PACKED B tile live in three LDS stages; tile kb+3 travels global -> registers and tile kb+2
//     registers -> LDS while tile kb is multiplied, and the operands of every MFMA step are
//     fetched (and decoded) one step ahead, across tile boundaries too;
//   * B is never materialised in memory at the compute type: lane (g, c) of a wave reads the
//     packed bytes of the half-tile k in [g*BK/2, (g+1)*BK/2) of its weight row and decodes them
//     in registers straight into MFMA operands.  The contraction index of MFMA step j is labelled
//     k = g*BK/2 + j*BK/8 + perm(e) for BOTH operands, where perm is whatever element order the
//     policy's cheapest decoder produces; the policy's A transform applies the same perm;
//   * A rows are 128 B in LDS, their 16-byte pieces XOR-swizzled with the row index so the 8
//     lanes of a ds_read_b128 phase hit 8 different bank groups;
//   * output tiles are assigned to workgroups so that each XCD (workgroup id mod 8) walks a
//     compact block of tiles and re-uses its A / B panels out of its own L2;
//   * the epilogue goes through LDS so that every lane stores 16 contiguous bytes (or, for the
//     transposed-output variants, contiguous runs along M).
#pragma once

#include "dq_common.h"
#include "dq_scale_walk.h"

#include <type_traits>

#ifndef DQ_SWZ_SHIFT
#define DQ_SWZ_SHIFT 1
#endif

namespace dq {
namespace gemm {

constexpr int BM = 256, BN = 256;
constexpr int kThreads = 256;
constexpr int kARowBytes = 128;            // bytes of one A row per k-block in LDS
constexpr int kAStage = BM * kARowBytes;   // 32 KiB

// XOR key of the 16-byte pieces of A row `row` in LDS (rows are 128 B).
__host__ __device__ constexpr int a_swz(int row) { return (row >> DQ_SWZ_SHIFT) & 7; }

// Where 16-byte piece `piece` of packed-B row `row` sits inside the row in LDS (register-staged kernel).  Rows of
// 32 or 64 bytes: rotated by the row index so that the 16 rows of one ds_read_b128 phase cover all 64 banks.  Rows
// of 128 bytes (an operand stored at the compute type, nothing to decode): the XOR swizzle of the A rows.
template <int kPieces>
__host__ __device__ constexpr int b_piece_pos(int row, int piece) {
  if (kPieces == 8) return piece ^ a_swz(row);
  return (piece + (row >> (kPieces == 2 ? 3 : 2))) % kPieces;
}

struct Params {
  const void* A;
  const void* B;
  const void* S;     // scales (policy specific) or nullptr
  const void* Z;     // zeros / second scale (policy specific) or nullptr
  const void* Bias;  // optional
  void* C;
  int M, N, K;       // K: contraction length of this launch (of one K slice when split > 1)
  int ldk;           // k elements per stored row of A and B (= K unless the launch covers K slices)
  int split;         // K slices, each its own set of workgroups and its own M x N output behind C
  int kunit;         // k per unit of which a slice is a run; read by policies with kUnevenSlices alone
  int tiles_m, tiles_n;
  int p0, p1;        // policy specific integers (e.g. scale exponent offset, group shift)
  float f0;          // policy specific float (e.g. 1 / weight scale)
};

// Workgroup id -> output tile.  With T tiles and 8 XCDs, XCD x (ids x, x+8, ...) gets a
// contiguous range of T/8 tiles, the first T%8 XCDs one more, of a sequence that walks the tile grid in bands of
// kGroupM tile rows, column by column inside a band.  (Up to 320 tiles that are no multiple of 8 go as they come (259: 26.9 us, sorted
// 28.9); beyond, sorted: MXFP4 M = 1316, N = 22608, K = 6912 385 -> 342 us, int8 x int4 M = 2217, N = 18000, K = 3328 155 -> 140.)
__device__ __forceinline__ void tile_of_block(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int T = tiles_m * tiles_n;
  int pid = bid;
  if ((T & 7) == 0 || T > 320) pid = (bid & 7) * (T >> 3) + min(bid & 7, T & 7) + (bid >> 3);
  constexpr int kGroupM = 4;
  const int band = kGroupM * tiles_n;
  const int first_m = (pid / band) * kGroupM;
  const int gm = min(tiles_m - first_m, kGroupM);
  const int in_band = pid - (pid / band) * band;
  tm = first_m + in_band % gm;
  tn = in_band / gm;
}

// P::kUnevenSlices: K slices as even as whole units of kunit k allow, instead of equal ones
template <class P, class = void>
struct UnevenSlices : std::false_type {};
template <class P>
struct UnevenSlices<P, std::void_t<decltype(P::kUnevenSlices)>> : std::integral_constant<bool, P::kUnevenSlices> {};

// Split-K (examples/dequantize_gemm/example_dequant_gemm_fp4_hopper.py:136-167): workgroup ids beyond the first
// tiles_m x tiles_n belong to further K slices.  Slice z reads columns [z K, (z + 1) K) of A and B, with uneven slices
// (where K comes in as all of ldk) the z-th of `split` runs of whole units, and writes the z-th M x N (or N x M) partial
// result behind C; a second kernel sums the partial results.  Plain (unpacked) A only.
template <class P>
__device__ __forceinline__ void take_k_slice(Params& p, int& bid) {
  if (p.split > 1) {
    const int tiles = p.tiles_m * p.tiles_n;
    const int z = bid / tiles;
    bid -= z * tiles;
    int k0 = z * p.K;
    if constexpr (UnevenSlices<P>::value) {
      const int units = p.ldk / p.kunit;
      const int u0 = units * z / p.split, u1 = units * (z + 1) / p.split;
      k0 = u0 * p.kunit;
      p.K = (u1 - u0) * p.kunit;
      // a slice starts where a dword of a row's scales does: kunit is a multiple of 128 k, and of two groups
      if constexpr (P::kScaleDma == 1) p.S = (const unsigned char*)p.S + (k0 >> 5);
      if constexpr (P::kScaleDma >= 2) p.S = (const unsigned char*)p.S + ((k0 >> p.p0) << 1);
      if constexpr (P::kScaleDma == 3) p.Z = (const unsigned char*)p.Z + ((k0 >> p.p0) << 1);
    }
    p.A = (const unsigned char*)p.A + (size_t)k0 * (kARowBytes / P::kKPerBlock);
    p.B = (const unsigned char*)p.B + (size_t)k0 * P::kBRowBytes / P::kKPerBlock;
    p.C = (unsigned char*)p.C + (size_t)z * p.M * p.N * sizeof(typename P::out_t);
  }
}

// Epilogue shared by both kernel variants (a macro: it uses the kernel's locals), over the first BLOCKS_ of the wave's kMBW
// blocks of rows.
// acc[mb][nb][i] = C[m0 + (wm*kMBW + mb)*32 + 8*(i/4) + 4*g + i%4][n0 + (wn*kNBW + nb)*32 + r], with kMBW x kNBW
// blocks of 32 x 32 per wave (constants of the kernel that expands the macro).  Staged through
// LDS (every tile is consumed: the loop ended with a barrier) so that each lane stores 16 contiguous
// bytes.  Each wave owns a slab of 32-bit values, 32 x (32 kNBW + 4) for a block of rows or, transposed, 32 x (32 kMBW + 4)
// for a block of columns; LDS operations of one wave execute in order, so no workgroup barrier is needed between the phases.
// The stores: C is written once and not read again by the kernel.  They are nontemporal, which keeps the output from
// displacing operand lines in the L2 (MXFP4 GEMM 361 -> 358 us, block-scaled GEMM 147 -> 138 us), except where a memory
// sector (32 bytes) is shared by two pieces, which a nontemporal store would each write to memory by itself: ordinary
// stores there, which meet in the L2 (int8 x 2-bit, M = 2048, N = 8200, K = 4096 118 -> 92 us, MXFP4 159 -> 140; with rows
// of whole sectors ordinary stores are the slower ones: M = 2664, N = 4560, K = 2304 39.8 against 44.6).  Columns of a
// transposed output, which other workgroups continue, take them where they are no whole cache lines (int8 x int4, M = 1000,
// N = 11008, K = 1024: 34 -> 21 us, nontemporal 24).  Which of the two is asked once per tile: asked per store it cost
// BitLinear at M = 2048, N = K = 8192 1 %.
// Transposed, the four consecutive rows that a lane holds are one LDS write.  A column that does not start at 16 bytes goes
// out by elements, consecutive lanes on consecutive elements, eight LDS reads ahead of their stores (a read under each store's
// condition waited for each: M = 1002, N = 11008, K = 1024 27.2 us, 23.6 so; M = 1001, K = 4096 58.4 and 53.8), or, where
// fewer than 48 rows are left, by blocks of 32 rows, a lane's four or eight one after the other (M = 3, N = 4448, K = 1024: 7.1
// us with all of the wave's rows walked, 6.3 so; M = 5, N = K = 4096 14.9 and 13.7).  Only the copy that needs them holds
// these forms: the wave fetches what it does not run too.
#define DQ_GEMM_EPILOGUE DQ_GEMM_EPILOGUE_OF(kMBW)
#define DQ_GEMM_EPILOGUE_OF(BLOCKS_) \
  if (P::kTransposed ? M * (int)sizeof(typename P::out_t) % 128 == 0 : N * (int)sizeof(typename P::out_t) % 32 == 0) { \
    DQ_GEMM_EPILOGUE_STORING(BLOCKS_, true) \
  } else { \
    DQ_GEMM_EPILOGUE_STORING(BLOCKS_, false) \
  }
#define DQ_GEMM_EPILOGUE_STORING(BLOCKS_, STREAMED_) \
  using out_t = typename P::out_t; \
  constexpr int kOutPerPiece = 16 / sizeof(out_t); \
  if constexpr (!P::kTransposed) { \
    constexpr int kSlabStride = 32 * kNBW + 4; \
    uint32_t* slab = reinterpret_cast<uint32_t*>(smem) + wave * (32 * kSlabStride); \
  _Pragma("unroll") \
    for (int mb = 0; mb < BLOCKS_; ++mb) { \
  _Pragma("unroll") \
      for (int nb = 0; nb < kNBW; ++nb) \
  _Pragma("unroll") \
        for (int i = 0; i < 16; ++i) { \
          const int row = 8 * (i >> 2) + 4 * g + (i & 3); \
          const decltype(acc[0][0][0] + 0) elem = acc[mb][nb][i]; \
          uint32_t bits; \
          __builtin_memcpy(&bits, &elem, 4); \
          slab[row * kSlabStride + nb * 32 + r] = bits; \
        } \
      __builtin_amdgcn_wave_barrier(); \
      constexpr int kPiecesPerRow = 32 * kNBW / kOutPerPiece; \
      constexpr int kIters = 32 * kPiecesPerRow / 64; \
  _Pragma("unroll") \
      for (int it = 0; it < kIters; ++it) { \
        const int q = lane + 64 * it; \
        const int row = q / kPiecesPerRow, piece = q % kPiecesPerRow; \
        const int m = m0 + wm * (32 * kMBW) + mb * 32 + row; \
        const int n = n0 + wn * (32 * kNBW) + piece * kOutPerPiece; \
        uint32_t raw[kOutPerPiece]; \
  _Pragma("unroll") \
        for (int e = 0; e < kOutPerPiece; e += 4) { \
          const uint4_t v = *reinterpret_cast<const uint4_t*>(slab + row * kSlabStride + piece * kOutPerPiece + e); \
          raw[e] = v[0]; raw[e + 1] = v[1]; raw[e + 2] = v[2]; raw[e + 3] = v[3]; \
        } \
        if (m < M && n < N) { \
          out_t o[kOutPerPiece]; \
  _Pragma("unroll") \
          for (int e = 0; e < kOutPerPiece; ++e) o[e] = P::finish(raw[e], p, m, min(n + e, N - 1)); \
          out_t* dst = (out_t*)p.C + (size_t)m * N + n; \
          if (STREAMED_ || (N % kOutPerPiece) == 0) { \
            uint4_t pk; \
            __builtin_memcpy(&pk, o, 16); \
            if constexpr (STREAMED_) __builtin_nontemporal_store(pk, reinterpret_cast<uint4_t*>(dst)); \
            else *reinterpret_cast<uint4_t*>(dst) = pk; \
          } else { \
  _Pragma("unroll") \
            for (int e = 0; e < kOutPerPiece; ++e) \
              if (n + e < N) dst[e] = o[e]; \
          } \
        } \
      } \
      __builtin_amdgcn_wave_barrier(); \
    } \
  } else { \
    constexpr int kRows = 32 * BLOCKS_; \
    constexpr int kSlabStride = kRows + 4; \
    uint32_t* slab = reinterpret_cast<uint32_t*>(smem) + wave * (32 * kSlabStride); \
    const int m_wave = m0 + wm * (32 * kMBW); \
    if (m_wave < M) \
  _Pragma("unroll") \
    for (int nb = 0; nb < kNBW; ++nb) { \
  _Pragma("unroll") \
      for (int mb = 0; mb < BLOCKS_; ++mb) \
  _Pragma("unroll") \
        for (int v = 0; v < 4; ++v) { \
          const decltype(acc[0][0][0] + 0) elem[4] = {acc[mb][nb][4 * v], acc[mb][nb][4 * v + 1], acc[mb][nb][4 * v + 2], acc[mb][nb][4 * v + 3]}; \
          uint4_t bits; \
          __builtin_memcpy(&bits, elem, 16); \
          *reinterpret_cast<uint4_t*>(slab + r * kSlabStride + mb * 32 + 8 * v + 4 * g) = bits; \
        } \
      __builtin_amdgcn_wave_barrier(); \
      const int n_block = n0 + wn * (32 * kNBW) + nb * 32; \
      if (STREAMED_ || (M % kOutPerPiece) == 0) { \
        constexpr int kPiecesPerCol = kRows / kOutPerPiece; \
  _Pragma("unroll") \
        for (int it = 0; it < 32 * kPiecesPerCol / 64; ++it) { \
          const int q = lane + 64 * it; \
          const int col = q / kPiecesPerCol, piece = q % kPiecesPerCol; \
          const int n = n_block + col, m = m_wave + piece * kOutPerPiece; \
          uint32_t raw[kOutPerPiece]; \
  _Pragma("unroll") \
          for (int e = 0; e < kOutPerPiece; e += 4) { \
            const uint4_t v = *reinterpret_cast<const uint4_t*>(slab + col * kSlabStride + piece * kOutPerPiece + e); \
            raw[e] = v[0]; raw[e + 1] = v[1]; raw[e + 2] = v[2]; raw[e + 3] = v[3]; \
          } \
          if (n < N && m < M) { \
            out_t o[kOutPerPiece]; \
  _Pragma("unroll") \
            for (int e = 0; e < kOutPerPiece; ++e) o[e] = P::finish(raw[e], p, m + e, n); \
            out_t* const dst = (out_t*)p.C + (size_t)n * M + m; \
            uint4_t pk; \
            __builtin_memcpy(&pk, o, 16); \
            if constexpr (STREAMED_) __builtin_nontemporal_store(pk, reinterpret_cast<uint4_t*>(dst)); \
            else *reinterpret_cast<uint4_t*>(dst) = pk; \
          } \
        } \
      } else if constexpr (!STREAMED_) { \
        if (M - m_wave < 48) { \
          constexpr int kPiecesPerCol = 32 / kOutPerPiece; \
  _Pragma("unroll") \
          for (int mb = 0; mb < BLOCKS_; ++mb) { \
            if (m_wave + 32 * mb >= M) break; \
  _Pragma("unroll") \
            for (int it = 0; it < kPiecesPerCol / 2; ++it) { \
              const int q = lane + 64 * it; \
              const int col = q / kPiecesPerCol, at = 32 * mb + q % kPiecesPerCol * kOutPerPiece; \
              const int n = n_block + col, m = m_wave + at; \
              uint32_t raw[kOutPerPiece]; \
  _Pragma("unroll") \
              for (int e = 0; e < kOutPerPiece; e += 4) { \
                const uint4_t v = *reinterpret_cast<const uint4_t*>(slab + col * kSlabStride + at + e); \
                raw[e] = v[0]; raw[e + 1] = v[1]; raw[e + 2] = v[2]; raw[e + 3] = v[3]; \
              } \
  _Pragma("unroll") \
              for (int e = 0; e < kOutPerPiece; ++e) \
                if (n < N && m + e < M) ((out_t*)p.C)[(size_t)n * M + m + e] = P::finish(raw[e], p, m + e, n); \
            } \
          } \
        } else { \
          constexpr int kBatch = 8; \
  _Pragma("unroll 1") \
          for (int it = 0; it < 32 * kRows / 64; it += kBatch) { \
            uint32_t raw[kBatch]; \
  _Pragma("unroll") \
            for (int u = 0; u < kBatch; ++u) { \
              const int q = lane + 64 * (it + u); \
              raw[u] = slab[q / kRows * kSlabStride + q % kRows]; \
            } \
  _Pragma("unroll") \
            for (int u = 0; u < kBatch; ++u) { \
              const int q = lane + 64 * (it + u); \
              const int m = m_wave + q % kRows, n = n_block + q / kRows; \
              if (n < N && m < M) ((out_t*)p.C)[(size_t)n * M + m] = P::finish(raw[u], p, m, n); \
            } \
          } \
        } \
      } \
      __builtin_amdgcn_wave_barrier(); \
    } \
  } \
  /* end of epilogue */

// Policy interface (all static):
//   kBRowBytes        packed B bytes per weight row per k-block: 32 or 64
//   kAPacked          A arrives as packed int4 (64 B per row per k-block, expanded while staging)
//   kKPerBlock        k values per block (64 for 16-bit operands, 128 for int8)
//   frag_t, acc_t     MFMA operand / accumulator vector types
//   mfma(a, b, c)
//   stage_a(uint4)    transform of one 16-byte A piece (16 B of one row) on its way to LDS
//   expand_a(uint4, uint4&, uint4&)   kAPacked only: 16 packed bytes -> two 16-byte pieces
//   ScaleRaw / Scale, fetch_scale(p, row, kb, g) / prep_scale(raw, p)
//   decode(const uint32_t* words, int j, const Scale&)  -> B operand of MFMA step j; `words` are
//       the lane's kBRowBytes/2 packed bytes as dwords
//   Epilogue: out_t, kTransposed, finish(acc value, p, m, n) -> value stored
// kKSplit = 2: eight waves, two per SIMD; waves 4..7 are a second copy of the pipeline (LDS stages of their own) that
// takes the odd k-blocks while waves 0..3 take the even ones, and hands its accumulators over once, through LDS,
// after the loop.  For problems that give each CU one small tile with a long K (BitNet at M = 256): the second wave
// of a SIMD runs its matrix instructions under the first one's decode and waits.  Needs an even number of k-blocks.
template <class P, int kMBW, int kNBW, int kKSplit = 1>
__global__ __launch_bounds__(kThreads * kKSplit, 1) void gemm_kernel(const Params p_in) {
  Params p = p_in;
  int bid = blockIdx.x;
  take_k_slice<P>(p, bid);
  extern __shared__ __align__(16) unsigned char smem_all[];
  static_assert(kKSplit == 1 || kKSplit == 2, "one or two copies of the pipeline");
  constexpr int BM = 64 * kMBW, BN = 64 * kNBW;  // 2 x 2 waves of kMBW x kNBW blocks of 32 x 32 (shadow the 256 x 256 default)
  constexpr int kAStage = BM * kARowBytes;
  constexpr int kBStage = BN * P::kBRowBytes;
  constexpr int kStage = kAStage + kBStage;
  constexpr int kBPiecesPerRow = P::kBRowBytes / 16;           // 2 or 4
  constexpr int kBPieces = BN * kBPiecesPerRow;                 // 16-byte pieces of a packed B tile
  constexpr int kBLoads = (kBPieces + kThreads - 1) / kThreads;
  constexpr int kBWords = P::kBRowBytes / 8;                    // dwords per lane: 4 or 8
  constexpr int kALoads = (P::kAPacked ? 4 : 8) * BM / 256;     // 16-byte global loads of A per thread

  const int tid = threadIdx.x & (kThreads - 1);
  const int kh = kKSplit == 1 ? 0 : (int)(threadIdx.x / kThreads);  // which copy of the pipeline
  unsigned char* const smem = smem_all + kh * (3 * kStage);
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;  // 2 x 2 waves
  const int g = lane >> 5, r = lane & 31;
  const int M = p.M, N = p.N, K = p.K;

  int tm, tn;
  tile_of_block(bid, p.tiles_m, p.tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int KB = K / P::kKPerBlock / kKSplit;  // k-blocks of this copy: kb -> global k-block kb * kKSplit + kh
  const size_t a_row_bytes = P::kAPacked ? (size_t)(p.ldk >> 1) : (size_t)p.ldk * (kARowBytes / P::kKPerBlock == 2 ? 2 : 1);
  const size_t b_row_bytes = (size_t)p.ldk * P::kBRowBytes / P::kKPerBlock;

  // ---- global -> register staging ---------------------------------------------------------
  // A piece q = tid + 256 i: row q / 8, 16-byte piece q % 8 of the 128-byte row.  A packed A row
  // is 64 B per block: piece q = tid + 256 i covers row q / 4, packed piece q % 4, and expands
  // to LDS pieces 2 (q % 4) and 2 (q % 4) + 1.
  const unsigned char* a_src[kALoads];
  int a_dst[kALoads], a_dst2[kALoads];
#pragma unroll
  for (int i = 0; i < kALoads; ++i) {
    const int q = tid + kThreads * i;
    if constexpr (P::kAPacked) {
      const int row = q >> 2, piece = q & 3;
      a_src[i] = (const unsigned char*)p.A + (size_t)min(m0 + row, M - 1) * a_row_bytes + piece * 16;
      a_dst[i] = row * 128 + (((2 * piece) ^ a_swz(row)) << 4);
      a_dst2[i] = row * 128 + (((2 * piece + 1) ^ a_swz(row)) << 4);
    } else {
      const int row = q >> 3, piece = q & 7;
      a_src[i] = (const unsigned char*)p.A + (size_t)min(m0 + row, M - 1) * a_row_bytes + piece * 16;
      a_dst[i] = row * 128 + ((piece ^ a_swz(row)) << 4);
      a_dst2[i] = 0;
    }
  }
  const unsigned char* b_src[kBLoads];
  int b_dst[kBLoads];
  bool b_on[kBLoads];  // a tile narrower than the workgroup leaves some threads without a piece
#pragma unroll
  for (int i = 0; i < kBLoads; ++i) {
    const int q0 = tid + kThreads * i;
    b_on[i] = q0 < kBPieces;
    const int q = b_on[i] ? q0 : 0;
    const int row = q / kBPiecesPerRow, piece = q % kBPiecesPerRow;
    b_src[i] = (const unsigned char*)p.B + (size_t)min(n0 + row, N - 1) * b_row_bytes + piece * 16;
    b_dst[i] = kAStage + row * P::kBRowBytes + (b_piece_pos<kBPiecesPerRow>(row, piece) << 4);
  }

  uint4_t a_reg[kALoads], b_reg[kBLoads];
  auto load_tile = [&](int kb_local) {
    const int kb = kb_local * kKSplit + kh;
    const size_t a_step = P::kAPacked ? 64 : 128;
#pragma unroll
    for (int i = 0; i < kALoads; ++i) a_reg[i] = *reinterpret_cast<const uint4_t*>(a_src[i] + (size_t)kb * a_step);
#pragma unroll
    for (int i = 0; i < kBLoads; ++i)
      if (b_on[i]) b_reg[i] = *reinterpret_cast<const uint4_t*>(b_src[i] + (size_t)kb * P::kBRowBytes);
  };
  auto store_tile = [&](int stage) {
    unsigned char* base = smem + stage * kStage;
#pragma unroll
    for (int i = 0; i < kALoads; ++i) {
      if constexpr (P::kAPacked) {
        uint4_t lo, hi;
        P::expand_a(a_reg[i], lo, hi);
        *reinterpret_cast<uint4_t*>(base + a_dst[i]) = lo;
        *reinterpret_cast<uint4_t*>(base + a_dst2[i]) = hi;
      } else {
        *reinterpret_cast<uint4_t*>(base + a_dst[i]) = P::stage_a(a_reg[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < kBLoads; ++i)
      if (b_on[i]) *reinterpret_cast<uint4_t*>(base + b_dst[i]) = b_reg[i];
  };

  // ---- fragment read offsets -----------------------------------------------------------------
  // A fragment of m-block mb, step j: row wm*128 + mb*32 + r, logical piece g*4 + j
  int a_row_off[kMBW], a_row_sw[kMBW];
#pragma unroll
  for (int mb = 0; mb < kMBW; ++mb) {
    const int row = wm * (32 * kMBW) + mb * 32 + r;
    a_row_off[mb] = row * 128;
    a_row_sw[mb] = a_swz(row);
  }
  // packed B of n-block nb: row wn*128 + nb*32 + r, the half of the row that belongs to group g
  int b_off[kNBW][kBWords / 4];
  int w_row[kNBW];
#pragma unroll
  for (int nb = 0; nb < kNBW; ++nb) {
    const int row = wn * (32 * kNBW) + nb * 32 + r;
    w_row[nb] = min(n0 + row, N - 1);
#pragma unroll
    for (int h = 0; h < kBPiecesPerRow / 2; ++h) {
      const int piece = g * (kBPiecesPerRow / 2) + h;
      b_off[nb][h] = kAStage + row * P::kBRowBytes + (b_piece_pos<kBPiecesPerRow>(row, piece) << 4);
    }
  }

  typename P::acc_t acc[kMBW][kNBW];
#pragma unroll
  for (int mb = 0; mb < kMBW; ++mb)
#pragma unroll
    for (int nb = 0; nb < kNBW; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0;

  // ---- fragment readers ---------------------------------------------------------------------
  using frag_t = typename P::frag_t;
  auto read_a = [&](const unsigned char* base, int j, frag_t (&af)[kMBW]) {
#pragma unroll
    for (int mb = 0; mb < kMBW; ++mb)
      af[mb] = *reinterpret_cast<const frag_t*>(base + a_row_off[mb] + ((((g << 2) + j) ^ a_row_sw[mb]) << 4));
  };
  auto read_b = [&](const unsigned char* base, uint32_t (&bw)[kNBW][kBWords]) {
#pragma unroll
    for (int nb = 0; nb < kNBW; ++nb)
#pragma unroll
      for (int h = 0; h < kBPiecesPerRow / 2; ++h) {
        const uint4_t v = *reinterpret_cast<const uint4_t*>(base + b_off[nb][h]);
        bw[nb][4 * h + 0] = v[0]; bw[nb][4 * h + 1] = v[1]; bw[nb][4 * h + 2] = v[2]; bw[nb][4 * h + 3] = v[3];
      }
  };

  // ---- prologue: tiles 0 and 1 in LDS, tile 2 in registers, fragments of (tile 0, step 0) ready --
  // Three LDS stages.  During iteration kb: tile kb+2 goes registers -> stage (kb+2)%3 (last read in
  // iteration kb-1, protected by the barrier that ended it), tile kb+3 goes global -> registers, tile
  // kb is multiplied out of stage kb%3, and during its last step the first fragments of tile kb+1 are
  // already fetched from stage (kb+1)%3 (written in iteration kb-1): one barrier per iteration and the
  // LDS -> register -> MFMA pipeline never drains.
  typename P::ScaleRaw sc_raw1[kNBW], sc_raw2[kNBW];  // raw scales of tiles kb+1 and kb+2
  typename P::Scale sc_c[kNBW], sc_n[kNBW];
  load_tile(0);
#pragma unroll
  for (int nb = 0; nb < kNBW; ++nb) {
    sc_c[nb] = P::prep_scale(P::fetch_scale(p, w_row[nb], kh, g), p);
    sc_raw1[nb] = P::fetch_scale(p, w_row[nb], (KB > 1 ? 1 : 0) * kKSplit + kh, g);
  }
  store_tile(0);
  if (KB > 1) {
    load_tile(1);
    store_tile(1);
  }
  if (KB > 2) load_tile(2);
  __syncthreads();

  uint32_t bw_c[kNBW][kBWords], bw_n[kNBW][kBWords];
  frag_t af_c[kMBW], bf_c[kNBW], af_n[kMBW], bf_n[kNBW];
  read_b(smem, bw_c);
  read_a(smem, 0, af_c);
#pragma unroll
  for (int nb = 0; nb < kNBW; ++nb) bf_c[nb] = P::decode(bw_c[nb], 0, sc_c[nb]);

  int stage = 0;
  for (int kb = 0; kb < KB; ++kb) {
    const int stage1 = stage == 2 ? 0 : stage + 1;
    const int stage2 = stage1 == 2 ? 0 : stage1 + 1;
    const unsigned char* base = smem + stage * kStage;
    const unsigned char* base_n = smem + stage1 * kStage;
    if (kb + 2 < KB) {
      store_tile(stage2);
#pragma unroll
      for (int nb = 0; nb < kNBW; ++nb) sc_raw2[nb] = P::fetch_scale(p, w_row[nb], (kb + 2) * kKSplit + kh, g);
    }
    if (kb + 3 < KB) load_tile(kb + 3);
    const bool has_next = kb + 1 < KB;

#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // fetch and decode the operands of the next step while this step's MFMAs run
      if (j < 3) {
        read_a(base, j + 1, af_n);
#pragma unroll
        for (int nb = 0; nb < kNBW; ++nb) bf_n[nb] = P::decode(bw_c[nb], j + 1, sc_c[nb]);
        if (j == 2 && has_next) read_b(base_n, bw_n);
      } else if (has_next) {
        read_a(base_n, 0, af_n);
#pragma unroll
        for (int nb = 0; nb < kNBW; ++nb) {
          sc_n[nb] = P::prep_scale(sc_raw1[nb], p);
          bf_n[nb] = P::decode(bw_n[nb], 0, sc_n[nb]);
        }
      }
#pragma unroll
      for (int mb = 0; mb < kMBW; ++mb)
#pragma unroll
        for (int nb = 0; nb < kNBW; ++nb) acc[mb][nb] = P::mfma(af_c[mb], bf_c[nb], acc[mb][nb]);
#pragma unroll
      for (int q = 0; q < kMBW; ++q) af_c[q] = af_n[q];
#pragma unroll
      for (int q = 0; q < kNBW; ++q) bf_c[q] = bf_n[q];
    }
#pragma unroll
    for (int nb = 0; nb < kNBW; ++nb) {
      sc_c[nb] = sc_n[nb];
      sc_raw1[nb] = sc_raw2[nb];
#pragma unroll
      for (int w = 0; w < kBWords; ++w) bw_c[nb][w] = bw_n[nb][w];
    }
    stage = stage1;
    __syncthreads();
  }

  if constexpr (kKSplit == 2) {
    // the second copy hands its accumulators to the first: [wave][mb][nb][lane] behind the epilogue's slabs
    constexpr int kSlabBytes = 4 * 32 * (32 * (kNBW > kMBW ? kNBW : kMBW) + 4) * 4;
    typename P::acc_t* red = reinterpret_cast<typename P::acc_t*>(smem_all + ((kSlabBytes + 63) & ~63)) + wave * (kMBW * kNBW * 64) + lane;
    if (kh == 1) {
#pragma unroll
      for (int mb = 0; mb < kMBW; ++mb)
#pragma unroll
        for (int nb = 0; nb < kNBW; ++nb) red[(mb * kNBW + nb) * 64] = acc[mb][nb];
    }
    __syncthreads();  // (the loop's last barrier already saw every wave done with the stages this area overlays)
    if (kh == 1) return;
#pragma unroll
    for (int mb = 0; mb < kMBW; ++mb)
#pragma unroll
      for (int nb = 0; nb < kNBW; ++nb) acc[mb][nb] = acc[mb][nb] + red[(mb * kNBW + nb) * 64];
  }
  {
    unsigned char* const smem = smem_all;  // the slabs of the epilogue start at the front
    DQ_GEMM_EPILOGUE
  }
}

// A policy may declare `static constexpr bool kBFragments = true`: its packed B was re-ordered offline into the
// matrix instruction's operand order, B[(N + 31) / 32][K / kKPerBlock][64 lanes][16 bytes] (lane 32 h + r of a
// block: bytes 16 h .. 16 h + 15 of that k-block of row r of the block of 32; 32-byte B rows only).  Read by the
// direct-to-LDS kernel: a B load is then 1 KiB contiguous and lands in LDS as the operand it is.
template <class P, class = void>
struct BFragments : std::false_type {};
template <class P>
struct BFragments<P, std::void_t<decltype(P::kBFragments)>> : std::integral_constant<bool, P::kBFragments> {};

// ---- direct-to-LDS variant ---------------------------------------------------------------------
// For policies whose A needs no transform on its way to LDS (any per-fragment transform is P::fix_a,
// applied after the fragment is read) and whose scales are absent, one byte per 32 k or one fp16 (plus
// one fp16 zero) per group of 32 to 4096 k (P::kScaleDma): the A and packed-B tiles, and the scales, travel
// global -> LDS with global_load_lds_dwordx4 / _dword, two tiles ahead of the MFMAs, without
// passing through registers.  A lane's 16 bytes land at LDS base + lane * 16 whatever its source
// address, so the XOR swizzle of the A rows is applied by permuting the SOURCE addresses.  These
// loads are issued from inline assembly and tracked by hand (one s_waitcnt vmcnt per tile): the
// kernel issues no other vector-memory load inside the main loop, so the counter only ever
// holds these.  Requires two k-blocks or more, whole ones, and A, B smaller than 4 GiB (32-bit lane offsets).
//
// M0 is written inside the statement and is not on its clobber list: clang treats M0 as a reserved register,
// warns that a reserved register on a clobber list "may not be preserved" and promises nothing for it.  What
// keeps this sound is that the statement sets M0 itself immediately before the one instruction that reads it,
// and that nothing else in these kernels depends on M0 across the statement: they use no other LDS-direct load,
// no GWS / sendmsg, no indirect register indexing and no v_readlane / v_writelane with M0 as the lane select,
// and gfx950 LDS instructions do not read M0 (that was the pre-gfx9 bounds clamp).
__device__ __forceinline__ void dma16(unsigned lds_addr, unsigned voff, const void* sbase) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\t" ::"s"(lds_addr), "v"(voff), "s"(sbase) : "memory");
}
__device__ __forceinline__ void dma4(unsigned lds_addr, unsigned voff, const void* sbase) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2\n\t" ::"s"(lds_addr), "v"(voff), "s"(sbase) : "memory");
}

// The same where `not_due` (wave-uniform) is zero.  The jump stays inside the statement: a branch of its own
// would cut the region that the scheduler spreads over the matrix instructions.
__device__ __forceinline__ void dma4_unless(int not_due, unsigned lds_addr, unsigned voff, const void* sbase) {
  asm volatile("s_cmp_lg_u32 %0, 0\n\ts_cbranch_scc1 .Lnot_due%=\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %2, %3\n.Lnot_due%=:" ::"s"(__builtin_amdgcn_readfirstlane(not_due)), "s"(lds_addr), "v"(voff), "s"(sbase) : "memory", "scc");
}

// Five forms, on a tile of 256 columns:
// * kMBW = 4, kNBW = 4, kWavesM = 2: 256 rows on 2 x 2 waves of 128 x 128, one workgroup per CU.
// * kMBW = 8, kNBW = 2, kWavesM = 1: 256 rows on four waves side by side, each 256 rows x 64 columns.  A wave then
//   decodes only the 64 weight rows it alone multiplies (with two rows of waves every packed word is decoded twice per
//   workgroup) and reads every A fragment of the tile instead: half the decode instructions, twice the LDS reads of A.
//   For policies whose decode keeps a lone wave's instruction issue busier than its matrix pipe (P::kTallWaves).
// * kMBW = 4, kNBW = 2, kWavesM = 1: 128 rows on four waves side by side of 128 x 64, for problems with too few tiles
//   of 256 rows.  With kKHalves = 2 on eight waves, two per SIMD: waves 4 .. 7 multiply the other half of every stage
//   (a second k-block, or with 64-byte rows of B the other two steps of the one k-block) into accumulators of their own,
//   and the two halves exchange sums through LDS before the epilogue, of which each does half.
// * kMBW = 3 and 6, kNBW = 2, kWavesM = 1: 96 rows, on four waves or (kKHalves = 2) eight, and 192 rows on four, as the two above:
//   for the policies with P::kRowCosts, where such tiles fill their rounds better.
// What bounds the 128-row form is the CU's load unit, which takes about two cycles per 64 bytes or per row piece, if that
// is shorter: with a 32-byte piece of B and a dword of scales and of zeros per weight row and k-block (two workgroups of
// four waves, 2 x 2) it was busy 87 % of the time and the matrix pipe 45 %.  So scales come only when their dword is due,
// a stage brings B in pieces of 64 bytes, and eight waves share one stage (load unit 45 %, matrix pipe 67 %).  fp16 x
// uint4 with zeros at M = 2048, N = 4096, K = 14336: 260 -> 233 (scales when due, waves side by side) -> 211 us; M = 300,
// N = 13824, K = 5120: 86 -> 73 -> 60; MXFP4 at M = 768, N = K = 8192, which stays on four waves (kOneOrder): 102 -> 92; int8 x
// 2-bit, M = 1024, N = K = 8192: 58 -> 53.5; int8 x int4, M = 1024, N = K = 8192: 64 -> 59.5.
//
// kOdd: K may be an odd number of k-blocks and a row's scale groups an odd number.  Both kinds are built: the one that asks is
// slower also where nothing is odd (MXFP4, M = 4096, N = K = 8192: 369 and 374 us; fp16 x uint4 at M = 2048, N = 4096,
// K = 14336 203 and 206, at M = 2015, N = 24640, K = 2048 191 and 193; int8 x 2-bit, M = 2048, N = K = 8192: 109.7 and 110.2).
template <class P, int kMBW, int kNBW, int kWavesM = 2, int kKHalves = 1, bool kOdd = false>
__global__ __launch_bounds__(256 * kKHalves, 32 * kMBW * kWavesM <= 128 ? 2 : 1) void gemm_kernel_dma(const Params p_in) {
  Params p = p_in;
  int bid = blockIdx.x;
  take_k_slice<P>(p, bid);
  extern __shared__ __align__(16) unsigned char smem[];
  static_assert(P::kBRowBytes == 32 || P::kBRowBytes == 64, "direct-to-LDS variant: 32 or 64 packed bytes per weight row per tile");
  static_assert(kWavesM == 2 ? (kMBW == 4 && kNBW == 4) : (kWavesM == 1 && (kMBW == 3 || kMBW == 4 || kMBW == 6 || kMBW == 8) && kNBW == 2), "one of the forms");
  static_assert(kKHalves == 1 || (kKHalves == 2 && kWavesM == 1 && kMBW <= 4), "two halves of a stage: 96 or 128 rows");
  constexpr int kWavesN = 8 / kNBW;            // waves across the 256 tile columns
  constexpr int kWaves = 4;                    // of one half
  constexpr int BM = 32 * kMBW * kWavesM;      // shadows the 256-row default
  constexpr bool kHalves = kKHalves == 2;
  constexpr int kStageTiles = kHalves && P::kBRowBytes == 32 ? 2 : 1;  // k-blocks in a stage
  constexpr int kSteps = kHalves && P::kBRowBytes == 64 ? 2 : 4;       // of a wave in a k-block
  constexpr int kAStage = BM * kARowBytes * kStageTiles;  // 32 KiB (16 for 128 rows and one k-block)
  constexpr int kDmaWaves = kWaves * kKHalves;
  constexpr int kAOps = BM * kStageTiles / 8 / kDmaWaves;  // A DMA instructions per wave per stage
  constexpr int kBPiecesPerRow = P::kBRowBytes / 16;          // 2 or 4
  constexpr bool kBFrag = BFragments<P>::value;
  constexpr int kBLoadPieces = kBPiecesPerRow * kStageTiles;  // of a row in one stage
  constexpr int kBRot = kBLoadPieces == 2 ? 3 : 2;            // piece rotation advances every 8 or 4 rows
  constexpr int kBOps = BN * kBPiecesPerRow * kStageTiles / 64 / kDmaWaves;    // packed-B DMA instructions per wave per tile
  constexpr int kBStage = BN * P::kBRowBytes * kStageTiles;  // 8 or 16 KiB
  constexpr int kStage = kAStage + kBStage;
  constexpr int kStages = 3;
  // A packed-B row of one tile is 32 bytes, a quarter of a cache line, and the next tile's row is the next 32:
  // the B loads of tiles t and t + 1 (t even) are issued as pairs, the same instruction for t and then for t + 1,
  // which halves the lines the B stream asks the L2 for.  Tile t + 1 then lands three iterations before it is
  // read, which takes a fourth B slot, so B gets a ring of its own behind the three A stages: kPairB.  (One 64-byte piece
  // of a row for both tiles, half the load unit's steps: 357.3 -> 357.8 us for MXFP4 at M = 4096, N = K = 8192, which the
  // load unit does not bind.)  Policies with 64-byte rows keep A and B side by side in three stages (a fourth 16 KiB
  // slot would not fit).
  constexpr bool kPairB = P::kBRowBytes == 32 && BM == 256;
  constexpr int kBRing = kPairB ? kStages * kAStage : kAStage;       // where B of slot 0 starts
  constexpr int kBSlot = kPairB ? kBStage : kStage;                  // distance between B slots
  constexpr int kAStride = kPairB ? kAStage : kStage;                // distance between A stages
  // Scales that travel by DMA (P::kScaleDma): 1 = one byte per 32 k (a dword per row covers a pair of tiles),
  // 2 = one fp16 per group of 64 .. 4096 k (a dword per row covers two groups: four tiles at group 128), 3 = the same
  // for scales and for zeros.  A dword is asked for with the first tile it serves (and with the first tile of all).
  // Ring: 4 slots x 1 KiB (256 rows x one dword), a second ring for the zeros.
  constexpr int kRing = kPairB ? kStages * kAStage + 4 * kBStage : kStages * kStage;
  constexpr int kSOps = P::kScaleDma == 0 ? 0 : (P::kScaleDma == 3 ? 2 : 1);  // scale DMA instructions per wave per tile, at most
  constexpr int kBWords = P::kBRowBytes / 8 * kSteps / 4;   // dwords per lane and 32-row block: 4 or 8
  static_assert(!kBFrag || P::kBRowBytes == 32, "fragment-ordered B: 32-byte rows");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int dma_wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = kHalves ? dma_wave / kWaves : 0;  // which half of a stage the wave multiplies
  const int wave = kHalves ? dma_wave % kWaves : dma_wave;
  const int wm = wave / kWavesN, wn = wave % kWavesN;
  const int g = lane >> 5, r = lane & 31;
  const int M = p.M, N = p.N, K = p.K;

  int tm, tn;
  tile_of_block(bid, p.tiles_m, p.tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int KB = K / P::kKPerBlock / kStageTiles;  // tiles, or stages of two of them
  const unsigned lds0 = (unsigned)(size_t)smem;  // LDS byte address of the dynamic segment

  // ---- per-lane source offsets: LDS chunk c (16 bytes) of a tile <- which global 16 bytes --------
  unsigned a_voff[kAOps], b_voff[kBOps];
#pragma unroll
  for (int i = 0; i < kAOps; ++i) {
    const int c = (dma_wave * kAOps + i) * 64 + lane;  // A chunk: row c / 8 (of half c / 1024), physical piece c % 8
    const int row = (c >> 3) % BM, pp = c & 7;
    a_voff[i] = (unsigned)min(m0 + row, M - 1) * (unsigned)(p.ldk * (kARowBytes / P::kKPerBlock)) + (unsigned)((pp ^ a_swz(row)) << 4) +
                (unsigned)((c >> 3) / BM * kARowBytes);
  }
#pragma unroll
  for (int i = 0; i < kBOps; ++i) {
    const int c = (dma_wave * kBOps + i) * 64 + lane;  // B chunk: row c / pieces per row, physical piece c % pieces per row
    const int row = c / kBLoadPieces, pp = c % kBLoadPieces;
    // LDS position (piece + rotation) % pieces holds source piece `piece`
    b_voff[i] = (unsigned)min(n0 + row, N - 1) * (unsigned)(p.ldk * P::kBRowBytes / P::kKPerBlock) +
                (unsigned)(((pp - (row >> kBRot)) & (kBLoadPieces - 1)) << 4);
    if constexpr (kBFrag) {
      // instruction (wave, i) brings the 32-row block wave * kBOps + i of the tile: 1 KiB as stored, lane-linear
      // (a stage of two tiles: 2 KiB)
      const int at = dma_wave * kBOps + i;
      const int blk = min((n0 >> 5) + at / kStageTiles, ((N + 31) >> 5) - 1);
      b_voff[i] = (unsigned)blk * (unsigned)(p.ldk / P::kKPerBlock) * 1024u + (unsigned)(at % kStageTiles) * 1024u + (unsigned)lane * 16u;
    }
  }
  // fp16 scales (kScaleDma >= 2): one per 2^p0 k (p.p0 = 5 .. 12, the policy's dma_ok checks it), so a dword of a row
  // serves 2^s_ps tiles of 64 k.  Groups of 32 k (one tile per dword, the two k halves of a tile in different groups)
  // need the scales issued with every tile: not the kPairB form, which dma_eligible keeps them away from.  The two scale
  // bytes of a tile (kScaleDma == 1) are two bytes per 64 k, placed as a group of 64 k is
  const int s_gshift = P::kScaleDma >= 2 ? p.p0 : 6;
  const int s_ps = s_gshift - 5;
  const bool s_odd = kOdd && P::kScaleDma != 0 && ((p.ldk >> s_gshift) & 1) != 0;
  const int s_ahead = s_odd ? -(lane & 1) : 0;  // rows of a tile start at an even one
  const ScaleWalk walk((unsigned)min(n0 + (tid & 255), N - 1), (unsigned)(p.ldk >> s_gshift), s_odd);  // waves 4..7 repeat 0..3

  // One tile = kSOps + kAOps + kBOps DMA instructions per thread: first the scale dword(s) (row tid) if one is due,
  // then the A chunks, then the packed-B chunks.  Two halves: waves 0 .. 3 bring the scales and waves 4 .. 7 the zeros.
  // Two tiles of a stage share its dwords: no groups of 32 k there.
  constexpr int kTileOps = kSOps + kAOps + kBOps;
  auto issue_op = [&](int op, int kb, int stage, int b_tile = -1) {
    const unsigned sbase = lds0 + stage * kAStride;
    const unsigned bbase = lds0 + kBRing + (kPairB ? (kb & 3) : stage) * kBSlot;
    if (op < kSOps) {
      if constexpr (P::kScaleDma != 0) {
        const int quad = (kb * kStageTiles) >> s_ps;
        dma4_unless(kHalves && kh != op ? 1 : (kb * kStageTiles) & ((1 << s_ps) - 1),
                    lds0 + kRing + op * 4096 + (quad & 3) * 1024 + (wave & 3) * 256, walk.from(quad),
                    (const unsigned char*)(op == 0 ? p.S : p.Z) + (size_t)quad * 4);
      }
    } else if (op < kSOps + kAOps) {
      const int i = op - kSOps;
      dma16(sbase + (dma_wave * kAOps + i) * 1024, a_voff[i], (const unsigned char*)p.A + (size_t)kb * (128 * kStageTiles));
    } else {
      const int i = op - kSOps - kAOps;
      dma16(bbase + (dma_wave * kBOps + i) * 1024, b_voff[i], (const unsigned char*)p.B + (size_t)(b_tile < 0 ? kb : b_tile) * ((kBFrag ? 1024 : P::kBRowBytes) * kStageTiles));
    }
  };
  auto issue_first_scales = [&] {
    if constexpr (P::kScaleDma != 0) {
#pragma unroll
      for (int op = 0; op < kSOps; ++op)
        dma4_unless(s_odd && !(kHalves && kh != op) ? 0 : 1, lds0 + kRing + op * 4096 + 3 * 1024 + (wave & 3) * 256, walk.start, op == 0 ? p.S : p.Z);
    }
  };
  // DMA instructions of one tile that may be outstanding while the one before is waited for: the scales come first in a
  // tile and only with some tiles, so a wait that counts without them is right with and without them
  constexpr int kWaitOps = kTileOps - kSOps;

  // ---- fragment read offsets (same LDS geometry as the register-staged kernel) --------------------
  int a_row_off[kMBW], a_row_sw[kMBW], b_off[kNBW][kBWords / 4], s_off[kNBW];
#pragma unroll
  for (int mb = 0; mb < kMBW; ++mb) {
    const int row = wm * (32 * kMBW) + mb * 32 + r;
    a_row_off[mb] = row * 128 + (kStageTiles == 2 ? kh * (BM * kARowBytes) : 0);
    a_row_sw[mb] = a_swz(row);
  }
#pragma unroll
  for (int nb = 0; nb < kNBW; ++nb) {
    const int row = wn * (32 * kNBW) + nb * 32 + r;
#pragma unroll
    for (int h = 0; h < kBWords / 4; ++h) {
      const int piece = (kStageTiles == 2 ? kh * kBPiecesPerRow : 0) + g * (kBPiecesPerRow / 2) + (kSteps == 2 ? kh : h);
      b_off[nb][h] = row * (16 * kBLoadPieces) + (((piece + (row >> kBRot)) & (kBLoadPieces - 1)) << 4);  // in its B slot
      // fragment order: block row / 32 of the tile, then the lanes as the matrix instruction numbers them
      if constexpr (kBFrag) b_off[nb][h] = (row >> 5) * (1024 * kStageTiles) + (kStageTiles == 2 ? kh * 1024 : 0) + lane * 16;
    }
    s_off[nb] = kRing + row * 4 + (P::kScaleDma == 1 ? g : (P::kScaleDma >= 2 && s_gshift == 5 ? 2 * g : 0));
  }
  using frag_t = typename P::frag_t;
  auto read_a1 = [&](const unsigned char* base, int j, int mb) -> frag_t {
    return P::fix_a(*reinterpret_cast<const frag_t*>(base + a_row_off[mb] + ((((g << 2) + (kSteps == 2 ? 2 * kh : 0) + j) ^ a_row_sw[mb]) << 4)));
  };
  // 32 rows further down the rotation of the packed-B pieces repeats ((32 >> kBRot) % kBPiecesPerRow == 0)
  // and the scale rows are 4 bytes apart: block nb sits at a constant distance from block 0, so one
  // address per tile serves all kNBW reads through their immediate offsets
  static_assert((32 >> kBRot) % kBLoadPieces == 0, "B rotation must repeat every 32 rows");
  auto read_b1 = [&](const unsigned char* base, int nb, uint32_t (&bw)[kBWords]) {
#pragma unroll
    for (int h = 0; h < kBWords / 4; ++h) {
      const uint4_t v = *reinterpret_cast<const uint4_t*>(base + b_off[0][h] + nb * (32 * 16 * kBLoadPieces));
      bw[4 * h + 0] = v[0]; bw[4 * h + 1] = v[1]; bw[4 * h + 2] = v[2]; bw[4 * h + 3] = v[3];
    }
  };
  // where the scale of 64-k tile kb lies from s_off on (groups of 32 k: the lane's half of the tile is in s_off)
  auto scale_at = [&](int kb) -> int {
    const int group = (kb << 6) >> s_gshift;
    const int aligned = ScaleWalk::aligned(group);
    if constexpr (!kOdd) return aligned;
    return aligned + ((ScaleWalk::one_ahead(group) - aligned) & s_ahead);
  };
  // the LDS read of a scale and the arithmetic on it are separate steps, so that the read can be issued a
  // chunk ahead of its first use
  auto read_scale_byte = [&](int step_kb, int nb) -> int {
    const int kb = step_kb * kStageTiles + (kStageTiles == 2 ? kh : 0);
    if constexpr (P::kScaleDma == 1) return (smem + s_off[0] + scale_at(kb))[nb * 128];
    else return 0;
  };
  auto read_scale1 = [&](int step_kb, int nb) -> typename P::Scale {
    const int kb = step_kb * kStageTiles + (kStageTiles == 2 ? kh : 0);  // the 64-k tile
    if constexpr (P::kScaleDma >= 2) {
      const unsigned char* at = smem + s_off[0] + scale_at(kb) + nb * 128;
      return P::ring_scale(at, at + 4096);
    } else {
      return P::prep_scale(read_scale_byte(kb, nb), p);
    }
  };

  typename P::acc_t acc[kMBW][kNBW];
#pragma unroll
  for (int mb = 0; mb < kMBW; ++mb)
#pragma unroll
    for (int nb = 0; nb < kNBW; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0;

  // ---- prologue: tiles 0 and 1 (and their scales) in flight; only tile 0 has to have landed -------
  issue_first_scales();
  if constexpr (kPairB) {  // scales, A of tile 0, the B pairs of tiles 0 and 1, then A of tile 1
#pragma unroll
    for (int op = 0; op < kSOps + kAOps; ++op) issue_op(op, 0, 0);
#pragma unroll
    for (int i = 0; i < kBOps; ++i) {
      issue_op(kSOps + kAOps + i, 0, 0);
      issue_op(kSOps + kAOps + i, 1, 1);
    }
#pragma unroll
    for (int op = kSOps; op < kSOps + kAOps; ++op) issue_op(op, 1, 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kAOps) : "memory");
  } else {
#pragma unroll
    for (int op = 0; op < kTileOps; ++op) issue_op(op, 0, 0);
#pragma unroll
    for (int op = 0; op < kTileOps; ++op) issue_op(op, 1, 1);  // KB >= 2
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kWaitOps) : "memory");
  }
  __syncthreads();

  typename P::Scale sc_c[kNBW];
  uint32_t bw_c[kNBW][kBWords];
  frag_t af_c[kMBW], bf_c[kNBW], af_n[kMBW], bf_n[kNBW];

  // One iteration = tile kb out of `stage`, as 16 chunks of 4 MFMAs (one A fragment against the four
  // B fragments) kept in order by scheduling barriers; every chunk carries side work that issues in
  // the shadow of its MFMAs.  The loop is skewed by one MFMA step so that nothing waits on LDS right
  // after the barrier:
  //   chunks  0..3   MFMAs of step 3 of tile kb-1 (operands already in registers); side work: read
  //                  the packed B words, the scales and the step-0 A fragments of tile kb, decode step 0
  //   chunks  4..15  MFMAs of steps 0..2 of tile kb; side work: read / decode the operands of the next
  //                  step (the step-3 operands stay in registers for the next iteration)
  //   chunks  0..10  also issue one DMA instruction each of tile kb+2 into stage (kb+2) % 3, which
  //                  was last read in iteration kb-1 and is free since the barrier that ended it.
  // Tile kb+2 is not read before iteration kb+2: its loads have almost two iterations to land.
  // A chunk with its side work cut into four pieces, one behind each of the chunk's four MFMAs, each piece
  // fenced by scheduling barriers: left to itself the scheduler issues one MFMA, then all of the side work
  // (about 50 cycles, longer than the 32 the MFMA runs), then the other three back to back, and the matrix
  // pipe idles once per chunk.
  auto chunk4 = [&](int q, auto do_mfma_tag, auto&& side_a, auto&& side_b, auto&& side_c, auto&& side_d) {
    constexpr bool do_mfma = decltype(do_mfma_tag)::value;
    if constexpr (do_mfma) acc[q][0] = P::mfma(af_c[q], bf_c[0], acc[q][0]);
    side_a();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (do_mfma) acc[q][1] = P::mfma(af_c[q], bf_c[1], acc[q][1]);
    side_b();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (do_mfma) acc[q][2] = P::mfma(af_c[q], bf_c[2], acc[q][2]);
    side_c();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (do_mfma) acc[q][3] = P::mfma(af_c[q], bf_c[3], acc[q][3]);
    side_d();
    __builtin_amdgcn_sched_barrier(0);
  };

  // odd_tag: tile kb is odd (only looked at with kPairB, where even iterations issue the B pairs of tiles
  // kb + 2 and kb + 3, the scales and A of tile kb + 2, and odd iterations A of tile kb + 2 only)
  auto iteration = [&](int kb, int stage, auto first_tag, auto next2_tag, auto odd_tag) {
    constexpr bool first = decltype(first_tag)::value;
    constexpr bool has_next2 = decltype(next2_tag)::value;
    constexpr bool odd = decltype(odd_tag)::value;
    const int stage2 = stage == 0 ? 2 : stage - 1;  // (stage + 2) % 3
    const unsigned char* base = smem + stage * kAStride;
    const unsigned char* bbase = smem + kBRing + (kPairB ? (kb & 3) : stage) * kBSlot;
    constexpr int kIterOps = !kPairB ? kTileOps : (odd ? kAOps : kSOps + kAOps + 2 * kBOps);  // issued per iteration at most
    // waves side by side: a step is one scheduling region of at most eight matrix instructions, or two
    constexpr int kRegions = kMBW > 4 ? 2 : 1, kRegionRows = kMBW / kRegions;
    constexpr int kPlaces = kWavesM == 2 ? 1 : (kIterOps <= 2 * kSteps * kRegions ? 2 : 3);  // for loads, in a region
    static_assert(kIterOps <= (kWavesM == 2 ? 16 : kPlaces * kSteps * kRegions), "more loads than the iteration has places for");
    {
      using DoMfma = std::integral_constant<bool, !first>;
      auto dma = [&](int chunk) {
        if constexpr (!kPairB) {
          if (has_next2 && chunk < kTileOps) issue_op(chunk, kb + 2, stage2);
        } else if constexpr (odd) {
          if (has_next2 && chunk < kAOps) issue_op(kSOps + chunk, kb + 2, stage2);
        } else {
          if (has_next2 && chunk < kSOps + kAOps) issue_op(chunk, kb + 2, stage2);
          else if (has_next2 && chunk < kIterOps) {
            const int j = chunk - kSOps - kAOps;  // B instruction j / 2 of tile kb + 2 + j % 2
            // (an odd count of tiles: the last pair's second half is asked for in the first one's place and never read)
            issue_op(kSOps + kAOps + (j >> 1), kb + 2 + (j & 1), stage2, kOdd ? min(kb + 2 + (j & 1), KB - 1) : -1);
          }
        }
      };
      int sc_byte[4];  // scale bytes are read in chunk 0 and turned into multipliers in chunk 1
      auto fetch_b = [&](int nb) {
        read_b1(bbase, nb, bw_c[nb]);
        if constexpr (P::kScaleDma >= 2) sc_c[nb] = read_scale1(kb, nb);
        else sc_byte[nb] = read_scale_byte(kb, nb);
      };
      auto finish_scale = [&](int nb) {
        if constexpr (P::kScaleDma < 2) sc_c[nb] = P::prep_scale(sc_byte[nb], p);
      };
      auto nothing = [] {};
      if constexpr (kWavesM == 1) {
        // A region's matrix instructions (its A fragments against the wave's two B fragments) and their side work, as a
        // pipeline of one matrix instruction, at most one LDS read and a few vector instructions: the fewer rows share a
        // decoded fragment, the more.  Skewed by one step like the 2 x 2 form below.
        constexpr int kValu = kMBW >= 6 ? 3 : kMBW == 4 ? 4 : 5;
        auto region = [&](int q0, auto do_mfma_tag, auto&& side) {
          if constexpr (decltype(do_mfma_tag)::value) {
#pragma unroll
            for (int q = 0; q < kRegionRows; ++q)
#pragma unroll
              for (int nb = 0; nb < 2; ++nb) acc[q0 + q][nb] = P::mfma(af_c[q0 + q], bf_c[nb], acc[q0 + q][nb]);
          }
          side();
#pragma unroll
          for (int q = 0; q < 2 * kRegionRows; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        auto read_rows = [&](int j, int q0) {
#pragma unroll
          for (int q = q0; q < q0 + kRegionRows; ++q) af_n[q] = read_a1(base, j, q);
        };
        auto loads = [&](int region_of_iteration) {
#pragma unroll
          for (int i = 0; i < kPlaces; ++i) dma(region_of_iteration * kPlaces + i);
        };
        auto first_operands = [&] {
          finish_scale(0);
          finish_scale(1);
          bf_n[0] = P::decode(bw_c[0], 0, sc_c[0]);
          bf_n[1] = P::decode(bw_c[1], 0, sc_c[1]);
        };
        if constexpr (kRegions == 1) {
          region(0, DoMfma{}, [&] {
            fetch_b(0);
            fetch_b(1);
            read_rows(0, 0);
            loads(0);
            first_operands();
          });
        } else {
          region(0, DoMfma{}, [&] {
            fetch_b(0);
            fetch_b(1);
            loads(0);
            read_rows(0, 0);
          });
          region(kRegionRows, DoMfma{}, [&] {
            read_rows(0, kRegionRows);
            loads(1);
            first_operands();
          });
        }
#pragma unroll
        for (int q = 0; q < kMBW; ++q) af_c[q] = af_n[q];
        bf_c[0] = bf_n[0];
        bf_c[1] = bf_n[1];
#pragma unroll
        for (int j = 0; j < kSteps - 1; ++j) {
          if constexpr (kRegions == 1) {
            region(0, std::true_type{}, [&] {
              read_rows(j + 1, 0);
              loads(j + 1);
              bf_n[0] = P::decode(bw_c[0], j + 1, sc_c[0]);
              bf_n[1] = P::decode(bw_c[1], j + 1, sc_c[1]);
            });
          } else {
            region(0, std::true_type{}, [&] {
              read_rows(j + 1, 0);
              loads(2 * j + 2);
              bf_n[0] = P::decode(bw_c[0], j + 1, sc_c[0]);
            });
            region(kRegionRows, std::true_type{}, [&] {
              read_rows(j + 1, kRegionRows);
              loads(2 * j + 3);
              bf_n[1] = P::decode(bw_c[1], j + 1, sc_c[1]);
            });
          }
#pragma unroll
          for (int q = 0; q < kMBW; ++q) af_c[q] = af_n[q];
          bf_c[0] = bf_n[0];
          bf_c[1] = bf_n[1];
        }
      } else {
      chunk4(0, DoMfma{}, [&] { fetch_b(0); fetch_b(1); }, [&] { dma(0); }, [&] { fetch_b(2); fetch_b(3); },
             [&] { af_n[0] = read_a1(base, 0, 0); });
      chunk4(1, DoMfma{}, [&] { af_n[1] = read_a1(base, 0, 1); finish_scale(0); }, [&] { dma(1); },
             [&] { af_n[2] = read_a1(base, 0, 2); finish_scale(1); }, [&] { finish_scale(2); });
      chunk4(2, DoMfma{}, [&] { af_n[3] = read_a1(base, 0, 3); finish_scale(3); }, [&] { dma(2); },
             [&] { bf_n[0] = P::decode(bw_c[0], 0, sc_c[0]); }, [&] { bf_n[1] = P::decode(bw_c[1], 0, sc_c[1]); });
      chunk4(3, DoMfma{}, [&] { bf_n[2] = P::decode(bw_c[2], 0, sc_c[2]); }, [&] { dma(3); },
             [&] { bf_n[3] = P::decode(bw_c[3], 0, sc_c[3]); }, nothing);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        af_c[q] = af_n[q];
        bf_c[q] = bf_n[q];
      }
#pragma unroll
      for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          chunk4(q, std::true_type{}, [&] { af_n[q] = read_a1(base, j + 1, q); }, [&] { dma(4 + j * 4 + q); },
                 [&] { bf_n[q] = P::decode(bw_c[q], j + 1, sc_c[q]); }, nothing);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          af_c[q] = af_n[q];
          bf_c[q] = bf_n[q];
        }
      }
      }
    }
    // tile kb+1 must have landed before the next iteration reads it; tile kb+2 (issued during this
    // iteration) may still be in flight
    if (has_next2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(!kPairB || !odd ? kIterOps - kSOps : kIterOps) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };

  // tiles come in (even, odd) pairs, an odd count ends with an even one
  using T = std::true_type;
  using F = std::false_type;
  int stage = 0;
  int kb = 0;
  auto next_stage = [&] { stage = stage == 2 ? 0 : stage + 1; };
  if constexpr (kHalves) {  // KB >= 3, any number
    iteration(0, 0, T{}, T{}, F{});
    stage = 1;
    for (kb = 1; kb + 2 < KB; ++kb) {
      iteration(kb, stage, F{}, T{}, F{});
      next_stage();
    }
    iteration(kb, stage, F{}, F{}, F{});  // kb = KB - 2
    next_stage();
    iteration(kb + 1, stage, F{}, F{}, F{});
  } else if (KB > 2) {
    iteration(0, 0, T{}, T{}, F{});
    stage = 1;
    for (kb = 1; kb + 3 < KB; kb += 2) {
      iteration(kb, stage, F{}, T{}, T{});
      next_stage();
      iteration(kb + 1, stage, F{}, T{}, F{});
      next_stage();
    }
    const bool odd_count = kOdd && (KB & 1) != 0;
    if (!odd_count) {
      iteration(kb, stage, F{}, T{}, T{});  // kb = KB - 3
      next_stage();
      iteration(++kb, stage, F{}, F{}, F{});
      next_stage();
      ++kb;
    }
    iteration(kb, stage, F{}, F{}, T{});
    if (odd_count) {
      next_stage();
      iteration(kb + 1, stage, F{}, F{}, F{});
    }
  } else {  // KB == 2
    iteration(0, 0, T{}, F{}, F{});
    iteration(1, 1, F{}, F{}, T{});
  }
  // step 3 of the last tile
#pragma unroll
  for (int q = 0; q < kMBW; ++q)
#pragma unroll
    for (int nb = 0; nb < kNBW; ++nb) acc[q][nb] = P::mfma(af_c[q], bf_c[nb], acc[q][nb]);

  if constexpr (kKHalves == 2) {
    // Each half hands its sums of the other's 32-row blocks over and finishes its own: [half][wave][block][nb][i / 4][lane]
    constexpr int kOwn0 = (kMBW + 1) / 2, kOwn1 = kMBW - kOwn0;  // blocks of the first half, of the second
    typedef decltype(acc[0][0][0] + 0) elem_t;
    typedef elem_t elem4_t __attribute__((ext_vector_type(4)));
    elem4_t* const red = reinterpret_cast<elem4_t*>(smem) + wave * (kOwn0 * 2 * 4 * 64) + lane;
    constexpr int kHalfPieces = 4 * kOwn0 * 2 * 4 * 64;
    auto hand_over = [&](auto first_block, auto blocks) {
      constexpr int q0 = decltype(first_block)::value;
#pragma unroll
      for (int q = 0; q < decltype(blocks)::value; ++q)
#pragma unroll
        for (int nb = 0; nb < kNBW; ++nb)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            red[kh * kHalfPieces + ((q * kNBW + nb) * 4 + v) * 64] =
                elem4_t{acc[q0 + q][nb][4 * v], acc[q0 + q][nb][4 * v + 1], acc[q0 + q][nb][4 * v + 2], acc[q0 + q][nb][4 * v + 3]};
    };
    auto take = [&](auto blocks) {
#pragma unroll
      for (int q = 0; q < decltype(blocks)::value; ++q)
#pragma unroll
        for (int nb = 0; nb < kNBW; ++nb)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const elem4_t other = red[(1 - kh) * kHalfPieces + ((q * kNBW + nb) * 4 + v) * 64];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[q][nb][4 * v + e] += other[e];
          }
    };
    using Own0 = std::integral_constant<int, kOwn0>;
    using Own1 = std::integral_constant<int, kOwn1>;
    if (kh == 0) {
      hand_over(Own0{}, Own1{});
    } else {
      hand_over(std::integral_constant<int, 0>{}, Own0{});
#pragma unroll
      for (int q = 0; q < kOwn1; ++q)
#pragma unroll
        for (int nb = 0; nb < kNBW; ++nb) acc[q][nb] = acc[q + kOwn0][nb];
    }
    __syncthreads();
    if constexpr (kOwn0 == kOwn1) {
      take(Own0{});
    } else {
      if (kh == 0) take(Own0{});
      else take(Own1{});
    }
    __syncthreads();  // the epilogue's slabs lie where the sums were handed over
    const int first_row = m0 + 32 * kOwn0 * kh, slab_wave = wave + kWaves * kh;
    {
      const int m0 = first_row, wave = slab_wave;
      if constexpr (kOwn0 == kOwn1) {
        DQ_GEMM_EPILOGUE_OF(kOwn0)
      } else if (kh == 0) {
        DQ_GEMM_EPILOGUE_OF(kOwn0)
      } else {
        DQ_GEMM_EPILOGUE_OF(kOwn1)
      }
    }
  } else {
    DQ_GEMM_EPILOGUE
  }
}

template <class P, int kMBW = 4, int kNBW = 4, int kKSplit = 1>
int launch(Params p, hipStream_t stream) {
  constexpr int kTileM = 64 * kMBW, kTileN = 64 * kNBW;
  constexpr int kPipe = kKSplit * 3 * (kTileM * kARowBytes + kTileN * P::kBRowBytes);
  // epilogue staging, and behind it the accumulators the second copy of the pipeline hands over
  constexpr int kSlabs = ((4 * 32 * (32 * (kNBW > kMBW ? kNBW : kMBW) + 4) * 4 + 63) & ~63) + (kKSplit - 1) * 4 * kMBW * kNBW * 64 * 64;
  constexpr int kLds = kPipe > kSlabs ? kPipe : kSlabs;
  static_assert(kLds <= 160 * 1024, "LDS budget");
  p.tiles_m = (p.M + kTileM - 1) / kTileM;
  p.tiles_n = (p.N + kTileN - 1) / kTileN;
  auto kern = gemm_kernel<P, kMBW, kNBW, kKSplit>;
  static bool lds_limit_raised[kMaxDevices];
  if (raise_lds_limit<kLds>(kern, lds_limit_raised)) return -1;
  hipLaunchKernelGGL(kern, dim3(p.tiles_m * p.tiles_n * p.split), dim3(kThreads * kKSplit), kLds, stream, p);
  DQ_CHECK_HIP(hipGetLastError());
  return 0;
}

// Tile choice by how many workgroups the 256 CUs get: 256 x 256 when that already gives about one per
// CU, else 128 x 128, else 128 x 64 (a narrower N tile repeats the weight decode less than a
// narrower M tile would).
template <class P>
int launch_auto(const Params& p, hipStream_t stream) {
  auto tiles = [&](int bm, int bn) { return (long)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn) * p.split; };
  if (tiles(256, 256) >= 192) return launch<P, 4, 4>(p, stream);
  if (tiles(128, 128) >= 192) return launch<P, 2, 2>(p, stream);
  // at most about one small tile per CU and a long K: two copies of the pipeline per workgroup, on alternate
  // k-blocks (int8 x 2-bit at M = 256, N = K = 8192: 35 -> 28.5 us).  Integer accumulation only: there the order
  // of the K sum does not show, while a float result would no longer match the other tile shapes bit for bit.
  if constexpr (P::kBRowBytes <= 64 && std::is_same<typename P::acc_t, int16_t_>::value) {
    if (tiles(128, 64) <= 320 && (p.K / P::kKPerBlock) % 2 == 0 && p.K / P::kKPerBlock >= 8) return launch<P, 2, 1, 2>(p, stream);
  }
  return launch<P, 2, 1>(p, stream);
}

// Whether the direct-to-LDS kernel takes the problem at all
template <class P>
bool dma_takes(const Params& p) {
  // 32-bit lane offsets: A rows are 128 bytes per K block, packed B rows kBRowBytes
  const size_t a_bytes = (size_t)p.M * (p.ldk / P::kKPerBlock) * kARowBytes;
  const size_t b_bytes = (size_t)p.N * (p.ldk / P::kKPerBlock) * P::kBRowBytes;
  // an odd count of groups and an odd count of rows: the last row's last dword would reach two bytes beyond the scales
  const bool beyond = P::kScaleDma != 0 && p.N % 2 != 0 && ((p.ldk >> (P::kScaleDma >= 2 ? p.p0 : 6)) & 1) != 0;
  return P::dma_ok(p) && !beyond && p.K % P::kKPerBlock == 0 && p.K >= 2 * P::kKPerBlock && a_bytes < (1ull << 32) && b_bytes < (1ull << 32);
}

inline long tiles_of(const Params& p, int rows) { return (long)((p.M + rows - 1) / rows) * ((p.N + BN - 1) / BN) * p.split; }

// Rounds of 256 workgroups, one per CU.  The last one takes two thirds of a full round however few tiles it has, the rest by
// their share (a lone tile runs at a higher clock and has the caches to itself: fp16 x uint4, K = 4096, 270 tiles of 256
// rows 176 us, 256 of them 108).
inline double dma_rounds(long tiles) {
  const long full = tiles / 256, rest = tiles % 256;
  return (double)full + (rest ? 0.65 + 0.35 * (double)rest / 256.0 : 0.0);
}

// P::kPairWorkgroups: 257 to 512 tiles of 128 x 256 run as two workgroups of four waves per CU, not as rounds of eight waves,
// and up to K = 1024 also where 192 tiles of 256 rows or more would fill their rounds better: int8 x 2-bit there takes 0.77 of the
// time (median of 41 shapes; beyond, the tall tile is ahead or even).
template <class P, class = void>
struct PairWorkgroups : std::false_type {};
template <class P>
struct PairWorkgroups<P, std::void_t<decltype(P::kPairWorkgroups)>> : std::integral_constant<bool, P::kPairWorkgroups> {};

// 256 x 256 tiles, or 128 x 256.  A round of the first costs 1.85 of the second's (K = 8192: fp16 x uint4 215 and 116 us,
// MXFP4 180 and 98, int8 x int4 84 and 57), so what decides is how either fills its rounds (up to 128 of the first never).  Measured on both, fp16 x uint4
// with zeros, K = 4096: M = 700, N = 11008 75 us in tiles of 256 rows, 98 in tiles of 128; M = 1000 92 and 106; M = 600 76
// and 56; M = 1100, N = 13824 176 and 119; M = 1300, N = 8192 92 and 102; M = 1500, N = 28672 300 and 338.
template <class P>
bool dma_eligible(const Params& p) {
  // fp16 scales of groups of 32 k go with every tile: not with the pairwise issue of the 32-byte-row form of this tile
  const bool scales_per_tile = P::kScaleDma >= 2 && P::kBRowBytes == 32 && p.p0 == 5;
  const long tiles = tiles_of(p, 256);
  if (PairWorkgroups<P>::value && (tiles < 192 || (p.K <= 1024 && tiles_of(p, 128) <= 512))) return false;
  return !scales_per_tile && dma_takes<P>(p) && 1.85 * dma_rounds(tiles) <= dma_rounds(tiles_of(p, 128));
}

// Too few 256 x 256 tiles but at least `min_tiles` of 128 x 256: the same kernel on the half-height tile, which keeps the
// operands on the direct-to-LDS path.  Below that the register-staged kernel's smaller tiles (N = 11008, 86 tiles, K = 5120:
// int8 x int4 31.9 against 33.4 us).  The int8 x 2-bit policy gains from 160 tiles on only (N = 8192, K = 5120: 128 tiles
// 32 against 30.3 us, 256 tiles 36 against 45).
constexpr int kHalfTileMin = 96;

// An odd count of k-blocks, where the register-staged kernel's tiles of 128 x 128, two in place of one here, just fill their
// rounds and K is short: it stays ahead (us, there and here: int8 x int4 to 127 tiles and 16 k-blocks, M = 273, N = 8087, K = 640
// 11.7 and 15.3, 455 shapes 1.08 in the mean; the 16-bit operands to eight, M = 409, N = 5890, K = 320 9.7 and 11.7, 503 shapes
// 1.04; int8 x 2-bit at 193 to 256 tiles and to eight, M = 317, N = 17954, K = 640 21.4 and 26.8, 274 shapes 1.03).
template <class P>
bool odd_count_stays(const Params& p) {
  const int blocks = p.K / P::kKPerBlock;
  const long tiles = tiles_of(p, 128);
  if (blocks % 2 == 0) return false;
  constexpr bool kInt = std::is_same<typename P::acc_t, int16_t_>::value;
  if (kInt && P::kBRowBytes == 32) return tiles > 192 && tiles <= 256 && blocks <= 8;
  return tiles < 128 && blocks <= (kInt ? 16 : 8);
}
template <class P>
bool dma_half_eligible(const Params& p, int min_tiles = kHalfTileMin) {
  return !dma_eligible<P>(p) && dma_takes<P>(p) && tiles_of(p, 128) >= min_tiles && !odd_count_stays<P>(p);
}

template <class P, int kMBW, int kNBW, int kWavesM = 2, int kKHalves = 1, bool kOdd = false>
int launch_dma_tile(Params p, hipStream_t stream) {
  // uneven slices start and end on an even block and an even group; eight waves take any count of stages
  if constexpr (!kOdd && !UnevenSlices<P>::value && (kKHalves == 1 || P::kScaleDma != 0)) {
    const bool odd_blocks = kKHalves == 1 && p.K / P::kKPerBlock % 2 != 0;
    const bool odd_groups = P::kScaleDma != 0 && ((p.ldk >> (P::kScaleDma >= 2 ? p.p0 : 6)) & 1) != 0;
    if (odd_blocks || odd_groups) return launch_dma_tile<P, kMBW, kNBW, kWavesM, kKHalves, true>(p, stream);
  }
  constexpr int kWaves = 4;
  constexpr int kTileM = 32 * kMBW * kWavesM;
  constexpr bool kPairB = P::kBRowBytes == 32 && kTileM == 256;  // as in the kernel: a fourth B slot
  constexpr int kPipe = 3 * (kKHalves == 2 && P::kBRowBytes == 32 ? 2 : 1) * (kTileM * kARowBytes + BN * P::kBRowBytes) + (kPairB ? BN * P::kBRowBytes : 0) + 8 * 1024;
  // epilogue staging; with K in two halves the accumulators handed over before it
  constexpr int kSlabs = kKHalves == 1 ? kWaves * 32 * (32 * (kNBW > kMBW ? kNBW : kMBW) + 4) * 4 : 128 * 1024;
  constexpr int kLds = kPipe > kSlabs ? kPipe : kSlabs;
  p.tiles_m = (p.M + kTileM - 1) / kTileM;
  p.tiles_n = (p.N + BN - 1) / BN;
  static_assert(kLds <= 160 * 1024, "LDS budget");
  auto kern = gemm_kernel_dma<P, kMBW, kNBW, kWavesM, kKHalves, kOdd>;
  static bool lds_limit_raised[kMaxDevices];
  if (raise_lds_limit<kLds>(kern, lds_limit_raised)) return -1;
  hipLaunchKernelGGL(kern, dim3(p.tiles_m * p.tiles_n * p.split), dim3(64 * kWaves * kKHalves), kLds, stream, p);
  DQ_CHECK_HIP(hipGetLastError());
  return 0;
}

// P::kTallWaves: the four waves side by side (see the kernel)
template <class P, class = void>
struct TallWaves : std::false_type {};
template <class P>
struct TallWaves<P, std::void_t<decltype(P::kTallWaves)>> : std::integral_constant<bool, P::kTallWaves> {};

template <class P>
int launch_dma(const Params& p, hipStream_t stream) {
  if constexpr (TallWaves<P>::value) return launch_dma_tile<P, 8, 2, 1>(p, stream);
  else return launch_dma_tile<P, 4, 4>(p, stream);
}

// P::kOneOrder: a row's products are added in one order whatever the tile
template <class P, class = void>
struct OneOrder : std::false_type {};
template <class P>
struct OneOrder<P, std::void_t<decltype(P::kOneOrder)>> : std::integral_constant<bool, P::kOneOrder> {};

// Eight waves on the two halves of every stage: at least three stages, and no groups of 32 k (a dword of scales per tile).  Uncut
// only where K is long enough for the halves' exchange of sums and the one workgroup per CU, up to 1024 four waves are ahead or
// even: against four (us), int8 x int4, 97 to 256 tiles, K <= 1024 up to 1.06 times, K > 4096 0.97; fp16 x uint4, K <= 512 1.03,
// K > 4096 0.87, and beyond 512 tiles, where two workgroups of four waves fill each other's ends of tiles, K <= 1024 1.12 to 1.2,
// K <= 2048 1.06, K <= 4096 1.0.  (The slices of a cut K, one tile of 512 k and more each, were measured on eight.)
template <class P>
bool dma_halves_take(const Params& p) {
  if constexpr (OneOrder<P>::value) return false;
  if constexpr (PairWorkgroups<P>::value)
    if (tiles_of(p, 128) > 256 && tiles_of(p, 128) <= 512) return false;
  const int shortest = UnevenSlices<P>::value && p.split > 1 ? p.K / p.kunit / p.split * p.kunit : p.K;
  const int stage_k = P::kKPerBlock * (P::kBRowBytes == 32 ? 2 : 1);
  if (p.split == 1 && shortest <= (tiles_of(p, 128) > 512 ? 2048 : 1024)) return false;
  return shortest % stage_k == 0 && shortest / stage_k >= 3 && !(P::kScaleDma >= 2 && p.p0 == 5);
}

template <class P>
int launch_dma_half(const Params& p, hipStream_t stream) {
  if constexpr (!OneOrder<P>::value)
    if (dma_halves_take<P>(p)) return launch_dma_tile<P, 4, 2, 1, 2>(p, stream);
  return launch_dma_tile<P, 4, 2, 1>(p, stream);
}

// P::kRowCosts: what a call takes on tiles of 96, 128, 192 and 256 rows (us: start + rounds x (round + K / 1000 x per_k), rounds
// as dma_rounds counts them), for the policies that are built at 96 and 192 rows too.  Fitted over 70 shapes a policy (140 to
// 3500 rows, N 1500 to 28500, K 1024 to 14300), where they pick tiles that are 5 % (uint4, MXFP4) and 8 % (2-bit) faster in the
// mean than the better of 128 and 256 rows; 7 % slower in the worst (uint4).  They are taken where they save a twenty-fifth.
// int8 x int4 gains nothing (0.5 %) and stays with the two.
struct RowsCost {
  double start, round, per_k;
};
template <class P, class = void>
struct HasRowCosts : std::false_type {};
template <class P>
struct HasRowCosts<P, std::void_t<decltype(P::kRowCosts)>> : std::true_type {};

// The tile's rows, or 0: not a call of the direct-to-LDS kernel.
template <class P>
int dma_rows(const Params& p, int min_tiles = kHalfTileMin) {
  int rows = dma_eligible<P>(p) ? 256 : dma_half_eligible<P>(p, min_tiles) ? 128 : 0;
  if constexpr (HasRowCosts<P>::value) {
    if (!rows) return 0;
    constexpr int kHeights[4] = {96, 128, 192, 256};
    auto us = [&](int i) { return P::kRowCosts[i].start + dma_rounds(tiles_of(p, kHeights[i])) * (P::kRowCosts[i].round + P::kRowCosts[i].per_k * p.K * 1e-3); };
    // Scales and zeros of groups of 32 k go with every tile, on four waves: beyond 192 tiles of 96 rows and from 1024 k on the load
    // unit takes longer over those than the costs say (M = 461, N = 25216, K = 3072 104 us on 128 rows, 152 on 96; 143 shapes 1.02 in
    // the mean, to 192 tiles 190 shapes 0.94)
    // And twice the tiles of 128 rows (97 to 128 rows of C) where a tile does little but store rows of C that are off 16 bytes (MXFP4,
    // K < 2048, 420 shapes: 128 rows 0.94 of the time of 96, M = 101, N = 31779, K = 256 14.8 and 18.5 us; from 2048 k on, and with rows
    // of whole 16 bytes, 1.01 to 1.14).
    const bool twice = tiles_of(p, 96) >= 2 * tiles_of(p, 128) && p.K < 2048 && p.N % 8 != 0;
    const bool low = !(P::kScaleDma == 3 && p.p0 == 5 && p.K >= 1024 && tiles_of(p, 96) > 192) && !twice;
    double best = 0.96 * us(rows == 256 ? 3 : 1);
    for (int i = low ? 0 : 1; i < 3; ++i)
      if (kHeights[i] != rows && us(i) < best) best = us(i), rows = kHeights[i];
  }
  return rows;
}
template <class P>
int launch_dma_rows(const Params& p, int rows, hipStream_t stream) {
  if constexpr (HasRowCosts<P>::value) {
    if (rows == 192) return launch_dma_tile<P, 6, 2, 1>(p, stream);
    if (rows == 96) {
      if constexpr (!OneOrder<P>::value)
        if (dma_halves_take<P>(p)) return launch_dma_tile<P, 3, 2, 1, 2>(p, stream);
      return launch_dma_tile<P, 3, 2, 1>(p, stream);
    }
  }
  return launch_dma_half<P>(p, stream);
}

// The tile choice of every policy that can take the direct-to-LDS path: that kernel where the problem has tiles enough,
// else the register-staged kernel with the tile size launch_auto picks.
template <class P>
int launch_best(const Params& p, hipStream_t stream) {
  const int rows = dma_rows<P>(p);
  if (rows == 256) return launch_dma<P>(p, stream);
  if (rows) return launch_dma_rows<P>(p, rows, stream);
  return launch_auto<P>(p, stream);
}

// ---- K sliced over workgroups, fp32 sums in between --------------------------------------------------
// A few dozen to a few hundred rows: M x N gives a fraction of the CUs a tile of 128 x 256, and each of them then runs
// all of K at the rate of its ring (7 to 9 ns per k).  Sliced, the same tiles fill the chip; what it costs is the slices'
// sums (4 bytes an element and slice, written and read: 2.2 TB/s) and a second kernel (with the pipeline's start and end
// 8 us).  MXFP4, N = K = 8192: M = 96 64 -> 25.5 us, M = 384 90 -> 55.  The sums are added in an order of their own, so
// the cut form takes the eight waves that the uncut one (kOneOrder) may not.
// The policy with its accumulators stored as they are: one slice's partial result.
template <class P>
struct PartialSums : P {
  static constexpr bool kUnevenSlices = true;
  static constexpr bool kOneOrder = false;
  using out_t = float;
  __device__ static __forceinline__ out_t finish(uint32_t raw, const Params&, int, int) { return __builtin_bit_cast(float, raw); }
};

// C = out_t(parts[0] + parts[1] + ... (+ Bias)), the slices in that order.  count % 4 == 0.
template <class OUT, bool HAS_BIAS>
__global__ __launch_bounds__(256) void ksplit_sum_kernel(const float* __restrict__ parts, const OUT* __restrict__ bias,
                                                         OUT* __restrict__ C, size_t count, int split) {
  typedef OUT out4_t __attribute__((ext_vector_type(4)));
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= count) return;
  float4_t v = *reinterpret_cast<const float4_t*>(parts + i);
  for (int z = 1; z < split; ++z) v = v + *reinterpret_cast<const float4_t*>(parts + (size_t)z * count + i);
  if constexpr (HAS_BIAS) {
    const out4_t b = *reinterpret_cast<const out4_t*>(bias + i);
    v = v + float4_t{(float)b[0], (float)b[1], (float)b[2], (float)b[3]};
  }
  *reinterpret_cast<out4_t*>(C + i) = out4_t{(OUT)v[0], (OUT)v[1], (OUT)v[2], (OUT)v[3]};
}

// p: the whole problem.  1: a shape that the 128 x 256 direct-to-LDS tile or the cut does not take.
template <class P>
int launch_ksplit(Params p, void* parts, int split, hipStream_t stream) {
  if (split < 2 || !dma_takes<P>(p)) return 1;
  const size_t count = (size_t)p.M * p.N;
  p.kunit = 2 * P::kKPerBlock;
  if (P::kScaleDma >= 2 && (2 << p.p0) > p.kunit) p.kunit = 2 << p.p0;
  if (p.K % p.kunit != 0 || p.K / p.kunit < split || count % 4 != 0) return 1;
  p.split = split;
  using out_t = typename P::out_t;
  out_t* const C = (out_t*)p.C;
  p.C = parts;
  // tiles of 96 rows where they are no more than those of 128
  const bool low = (p.M + 95) / 96 == (p.M + 127) / 128;
  if (low ? launch_dma_rows<PartialSums<P>>(p, 96, stream) : launch_dma_half<PartialSums<P>>(p, stream)) return -1;
  const dim3 blocks((unsigned)((count + 1023) / 1024));
  if (p.Bias)
    hipLaunchKernelGGL((ksplit_sum_kernel<out_t, true>), blocks, dim3(256), 0, stream, (const float*)parts, (const out_t*)p.Bias, C, count, split);
  else
    hipLaunchKernelGGL((ksplit_sum_kernel<out_t, false>), blocks, dim3(256), 0, stream, (const float*)parts, (const out_t*)nullptr, C, count, split);
  DQ_CHECK_HIP(hipGetLastError());
  return 0;
}

inline Params make_params(const void* A, const void* B, const void* S, const void* Z, const void* Bias, void* C, int M,
                          int N, int K) {
  Params p{};
  p.A = A; p.B = B; p.S = S; p.Z = Z; p.Bias = Bias; p.C = C;
  p.M = M; p.N = N; p.K = K;
  p.ldk = K;
  p.split = 1;
  p.tiles_m = (M + BM - 1) / BM;
  p.tiles_n = (N + BN - 1) / BN;
  return p;
}

// ---- building blocks shared by the policies -------------------------------------------------------

struct NoScale {
  static constexpr int kScaleDma = 0;  // no scales to bring in by DMA
  static bool dma_ok(const Params&) { return true; }
  struct ScaleRaw {};
  struct Scale {};
  __device__ static __forceinline__ ScaleRaw fetch_scale(const Params&, int, int, int) { return {}; }
  __device__ static __forceinline__ Scale prep_scale(ScaleRaw, const Params&) { return {}; }
};

struct PlainA {
  static constexpr bool kAPacked = false;
  static constexpr bool kPlainA = true;  // stage_a is the identity: A may go global -> LDS directly
  __device__ static __forceinline__ uint4_t stage_a(uint4_t v) { return v; }
  __device__ static __forceinline__ void expand_a(uint4_t, uint4_t&, uint4_t&) {}
  // direct-to-LDS kernel: transform of an A fragment after it is read from LDS (A lands untouched)
  template <class F>
  __device__ static __forceinline__ F fix_a(F f) { return f; }
};

}  // namespace gemm
}  // namespace dq
