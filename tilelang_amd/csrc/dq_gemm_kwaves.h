// Dequantize GEMM of a few dozen rows on gfx950: K over the waves of a workgroup.
//
// The tiled kernels of dq_gemm_core.h give M x N / (128 x 256) workgroups all of K each: at 64 rows of N = K = 8192 that is 32
// workgroups for 256 CUs.  Here a workgroup owns few columns (32 or 64 weight rows) and few activation rows (16 to 64: what it
// holds accumulators for, more run as passes), and its eight or four waves take an eighth or a quarter of K each:
//   * a wave is a pipeline of its own: 4 KiB of LDS per 32 activation rows and 32 weight rows, written and read by that wave
//     alone.  A wave's LDS operations are carried out in the order they were issued, so the loop over K has no barrier and the
//     two waves of a SIMD run into each other's waits;
//   * weights come a cache line of each row at a time (a chunk: four tiles of 64 k at 4 bits by 16, two of 128 k at 4 bits by 8,
//     four at 2 by 8), activations a line per row and tile.  Both land in registers (weights a chunk ahead, activations
//     two tiles ahead), go through the wave's LDS into the operand order of the matrix instruction, and are decoded as
//     in dq_gemm_core.h, by the same policies;
//   * scales of a row travel 16 bytes at a time (a window: eight groups, or 512 k of block exponents), from whatever byte they
//     lie at;
//   * the waves' sums of an output meet in LDS, a block of 32 activation rows at a time, and are added in slice order.
// What bounds it is the load unit and the LDS port of a CU, which take a byte of A and B once in and once out each: per tile
// of 64 k and wave (64 rows x 64 columns) 10 KiB in and 10 KiB out beside 16 matrix instructions.
#pragma once

#include "dq_gemm_core.h"

namespace dq {
namespace gemm {

// AL: activation rows / 8 that a workgroup loads (the accumulators are blocks of 32); NB: blocks of 32 weight rows.
template <class P, int AL, int NB, int kWaves>
__global__ __launch_bounds__(64 * kWaves, 2) void gemm_kernel_kwaves(const Params p) {
  extern __shared__ __align__(16) unsigned char smem[];
  static_assert(!P::kAPacked && (P::kBRowBytes == 32 || P::kBRowBytes == 64), "int8 or 16-bit activations");
  constexpr int MB = (AL + 3) / 4;
  constexpr int T = 128 / P::kBRowBytes;       // tiles in a chunk
  constexpr int kBWords = P::kBRowBytes / 8;   // dwords per lane, tile and block of 32 weight rows
  using frag_t = typename P::frag_t;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5, r = lane & 31;
  const int M = p.M, N = p.N;

  // Workgroups x, x + 8, ... share an XCD and its L2: the passes over one set of weight rows follow each other there.
  const int passes = p.tiles_m, j_in = (int)blockIdx.x >> 3;
  const int nt = j_in / passes * 8 + ((int)blockIdx.x & 7);
  if (nt >= p.tiles_n) return;
  const int m0 = j_in % passes * (8 * AL), n0 = nt * (32 * NB);

  // the wave's chunks; which part of K is its own turns with the workgroup, so that the CUs do not ask for the same
  // stretch of every row at once
  const int KT = p.K / P::kKPerBlock, NC = (KT + T - 1) / T;
  const int kw = (wave + (nt >> 3)) & (kWaves - 1);
  const int c0 = kw * NC / kWaves, c1 = (kw + 1) * NC / kWaves;
  const int t_last = min(c1 * T, KT) - 1;

  typename P::acc_t acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0;

  if (c0 < c1) {
    const unsigned a_row_bytes = (unsigned)(p.ldk * (kARowBytes / P::kKPerBlock)), b_row_bytes = (unsigned)(p.ldk / P::kKPerBlock * P::kBRowBytes);
    // Load i: rows 8 i .. 8 i + 7, whole lines, through buffer descriptors: rows beyond the matrix and tiles beyond the wave's
    // (a descriptor of no bytes) come as zeros, so every load is unconditional and the compiler's count of those in flight exact.
    unsigned a_voff[AL], b_voff[4 * NB];
#pragma unroll
    for (int i = 0; i < AL; ++i) a_voff[i] = (unsigned)(m0 + 8 * i + (lane >> 3)) * a_row_bytes + (lane & 7) * 16;
#pragma unroll
    for (int i = 0; i < 4 * NB; ++i) b_voff[i] = (unsigned)(n0 + 8 * i + (lane >> 3)) * b_row_bytes + (lane & 7) * 16;
    uint4_t a_reg[2][AL], b_reg[4 * NB];
    auto load16 = [&](const void* base, unsigned bytes, unsigned first, bool on, unsigned voff) __attribute__((always_inline)) {
      __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)((const unsigned char*)base + first), 0, on ? bytes - first : 0u, 0x00027000);
      return __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff, 0, 0));
    };
    auto load_a = [&](uint4_t (&a)[AL], int t) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < AL; ++i) a[i] = load16(p.A, (unsigned)M * a_row_bytes, (unsigned)t * kARowBytes, t <= t_last, a_voff[i]);
    };
    auto load_b = [&](int c) __attribute__((always_inline)) {  // (of a part of a chunk, the rest is the next row's)
#pragma unroll
      for (int i = 0; i < 4 * NB; ++i) b_reg[i] = load16(p.B, (unsigned)N * b_row_bytes, (unsigned)c * 128u, c < c1, b_voff[i]);
    };

    // ---- scales: the window of 16 bytes of each of the lane's rows
    constexpr bool kS = P::kScaleDma != 0, kZ = P::kScaleDma == 3;
    const int s_gshift = P::kScaleDma >= 2 ? p.p0 : 6;   // (two bytes per 64 k: see gemm_kernel_dma)
    const int s_row_bytes = kS ? p.ldk >> s_gshift << 1 : 0;
    const int s_wshift = s_gshift - 5;                    // chunks per window
    uint4_t s_cur[NB], s_nxt[NB], z_cur[NB], z_nxt[NB];
    typedef uint4_t uint4_any __attribute__((aligned(1)));
    auto load_scales = [&](uint4_t (&s)[NB], uint4_t (&z)[NB], int window) __attribute__((always_inline)) {
      if constexpr (kS) {
        const int at = min(16 * window, s_row_bytes - 16);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const size_t off = (size_t)min(n0 + 32 * nb + r, N - 1) * s_row_bytes + at;
          s[nb] = *reinterpret_cast<const uint4_any*>((const unsigned char*)p.S + off);
          if constexpr (kZ) z[nb] = *reinterpret_cast<const uint4_any*>((const unsigned char*)p.Z + off);
        }
      }
    };
    // (a tile beyond the wave's: a finite scale, whose products with the zeros of A are zeros)
    auto scale_of = [&](int t, int nb) __attribute__((always_inline)) -> typename P::Scale {
      if constexpr (kS) {
        const int window = (t / T) >> s_wshift;
        const int idx = ((t << 6) >> s_gshift) - min(16 * window, s_row_bytes - 16) / 2;  // 16-bit elements into the window
        auto pick = [&](uint4_t v) { return idx < 4 ? (idx < 2 ? v[0] : v[1]) : (idx < 6 ? v[2] : v[3]); };
        if constexpr (P::kScaleDma == 1) {
          const int e = (int)(pick(s_cur[nb]) >> ((idx & 1) * 16 + g * 8) & 0xFFu);
          return P::prep_scale(t <= t_last ? e : 127 - p.p0, p);
        } else {
          const int sh = s_gshift == 5 ? g * 16 : (idx & 1) * 16;
          typename P::ScaleRaw raw{};
          raw.s = __builtin_bit_cast(half_t, (unsigned short)(t <= t_last ? pick(s_cur[nb]) >> sh : 0u));
          if constexpr (kZ) raw.z = __builtin_bit_cast(half_t, (unsigned short)(t <= t_last ? pick(z_cur[nb]) >> sh : 0u));
          return P::prep_scale(raw, p);
        }
      } else {
        return P::prep_scale(0, p);
      }
    };

    // ---- the wave's LDS: MB x 4 KiB of A (one tile), NB x 4 KiB of B (one chunk); rows of 128 bytes, pieces swizzled
    unsigned char* const lds_a = smem + wave * ((MB + NB) * 4096);
    unsigned char* const lds_b = lds_a + MB * 4096;
    const int wr0 = (lane >> 3) * 128 + (((lane & 7) ^ a_swz(lane >> 3)) << 4), wr1 = (lane >> 3) * 128 + (((lane & 7) ^ a_swz(8 + (lane >> 3))) << 4);
    auto at_piece = [&](int piece) { return r * 128 + ((piece ^ a_swz(r)) << 4); };

    auto do_tile = [&](int t, int q, uint4_t (&a)[AL]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < AL; ++i) *reinterpret_cast<uint4_t*>(lds_a + i * 1024 + ((i & 1) ? wr1 : wr0)) = P::stage_a(a[i]);
      asm volatile("" ::: "memory");  // the writes above are read by other lanes
      load_a(a, t + 2);
      uint32_t bw[NB][kBWords];
      typename P::Scale sc[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
        for (int h = 0; h < kBWords / 4; ++h) {
          const uint4_t v = *reinterpret_cast<const uint4_t*>(lds_b + nb * 4096 + at_piece(q * (8 / T) + g * (kBWords / 4) + h));
          bw[nb][4 * h] = v[0], bw[nb][4 * h + 1] = v[1], bw[nb][4 * h + 2] = v[2], bw[nb][4 * h + 3] = v[3];
        }
        sc[nb] = scale_of(t, nb);
      }
      frag_t af[2][MB];  // a step's operands are read a step ahead
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) af[0][mb] = *reinterpret_cast<const frag_t*>(lds_a + mb * 4096 + at_piece(4 * g));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j < 3)
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) af[(j + 1) & 1][mb] = *reinterpret_cast<const frag_t*>(lds_a + mb * 4096 + at_piece(4 * g + j + 1));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const frag_t bf = P::decode(bw[nb], j, sc[nb]);
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) acc[mb][nb] = P::kTransposed ? P::mfma(af[j & 1][mb], bf, acc[mb][nb]) : P::mfma(bf, af[j & 1][mb], acc[mb][nb]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      asm volatile("" ::: "memory");
    };

    int window = c0 >> s_wshift;
    load_b(c0);
    load_scales(s_cur, z_cur, window);
    load_a(a_reg[0], c0 * T);
    load_a(a_reg[1], c0 * T + 1);
    for (int c = c0; c < c1; ++c) {
#pragma unroll
      for (int i = 0; i < 4 * NB; ++i) *reinterpret_cast<uint4_t*>(lds_b + i * 1024 + ((i & 1) ? wr1 : wr0)) = b_reg[i];
      asm volatile("" ::: "memory");
      const int next = min(c + 1, c1 - 1);
      const bool turn = kS && (next >> s_wshift) != window;
      if (turn) load_scales(s_nxt, z_nxt, next >> s_wshift);
      load_b(c + 1);
#pragma unroll
      for (int q = 0; q < T; ++q) do_tile(c * T + q, q, a_reg[q & 1]);
      if (turn) {
        window = next >> s_wshift;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) s_cur[nb] = s_nxt[nb], z_cur[nb] = z_nxt[nb];
      }
    }
  }

  // ---- the waves' sums: a block of 32 activation rows at a time, two buffers, one barrier per block.  A wave's sums are
  // rows of 128 NB bytes (an activation row's columns) or, transposed, of 128 (a column's activation rows).
  __syncthreads();  // every wave is done with its areas
  constexpr int kPart = 4096 * NB;
  typedef decltype(acc[0][0][0] + 0) elem_t;
  typedef elem_t elem4_t __attribute__((ext_vector_type(4)));
  constexpr int kPieces = P::kTransposed ? 8 : 8 * NB;  // of a row
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    unsigned char* const buf = smem + (mb & 1) * (kWaves * kPart);
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = P::kTransposed ? 32 * nb + r : r, piece = P::kTransposed ? 2 * v + g : 8 * nb + 2 * v + g;
        *reinterpret_cast<elem4_t*>(buf + kw * kPart + row * (16 * kPieces) + ((piece ^ (r & 7)) << 4)) =
            elem4_t{acc[mb][nb][4 * v], acc[mb][nb][4 * v + 1], acc[mb][nb][4 * v + 2], acc[mb][nb][4 * v + 3]};
      }
    __syncthreads();
#pragma unroll
    for (int f = tid; f < 256 * NB; f += 64 * kWaves) {
      const int f_row = f / kPieces, f_piece = f % kPieces;
      elem4_t sum = *reinterpret_cast<const elem4_t*>(buf + f_row * (16 * kPieces) + ((f_piece ^ (f_row & 7)) << 4));
#pragma unroll
      for (int w = 1; w < kWaves; ++w)
        sum = sum + *reinterpret_cast<const elem4_t*>(buf + w * kPart + f_row * (16 * kPieces) + ((f_piece ^ (f_row & 7)) << 4));
      const int m = m0 + 32 * mb + (P::kTransposed ? 4 * f_piece : f_row), n = n0 + (P::kTransposed ? f_row : 4 * f_piece);
      using out_t = typename P::out_t;
      typedef out_t out4_t __attribute__((ext_vector_type(4)));
      const int m_end = min(M, m0 + 8 * AL);
      if (m < m_end && n < N) {
        out_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const elem_t x = sum[e];
          uint32_t bits;
          __builtin_memcpy(&bits, &x, 4);
          o[e] = P::kTransposed ? P::finish(bits, p, min(m + e, M - 1), n) : P::finish(bits, p, m, min(n + e, N - 1));
        }
        out_t* const dst = (out_t*)p.C + (P::kTransposed ? (size_t)n * M + m : (size_t)m * N + n);
        const int left = P::kTransposed ? m_end - m : N - n;
        if (P::kTransposed ? (M & 3) == 0 : (N & 3) == 0) {
          *reinterpret_cast<out4_t*>(dst) = out4_t{o[0], o[1], o[2], o[3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (e < left) dst[e] = o[e];
        }
      }
    }
  }
}

// Whether the kernel takes the call at all
template <class P>
bool kwaves_takes(const Params& p) {
  const size_t a_bytes = (size_t)p.M * (p.ldk / P::kKPerBlock) * kARowBytes;
  const size_t b_bytes = (size_t)p.N * (p.ldk / P::kKPerBlock) * P::kBRowBytes;
  if (p.split != 1 || p.K % P::kKPerBlock != 0 || a_bytes >= (1ull << 32) || b_bytes >= (1ull << 32)) return false;
  if (P::kScaleDma == 1) return p.K >= 512;  // a row of scales holds a window
  if (P::kScaleDma >= 2) return p.p0 >= 5 && p.p0 <= 12 && (p.K >> p.p0) >= 8 && (((size_t)p.S | (size_t)p.Z) & 1) == 0;
  return true;
}

// The forms that are built: activation rows / 8 and blocks of 32 weight rows of a workgroup, its waves.
struct KwavesForm {
  int al, nb, waves;
};
constexpr KwavesForm kKwavesForms[] = {{2, 1, 8}, {4, 1, 8}, {4, 2, 4}, {6, 2, 4}, {8, 2, 4}};
constexpr int kKwavesFormCount = 5;

// Workgroups of a call: passes over the rows, each of whole groups of eight sets of weight rows (one per XCD)
inline long kwaves_workgroups(const KwavesForm& f, int M, int N) {
  const long passes = ((long)M + 8 * f.al - 1) / (8 * f.al), sets = ((long)N + 32 * f.nb - 1) / (32 * f.nb);
  return passes * ((sets + 7) / 8 * 8);
}

template <class P, int AL, int NB, int kWaves>
int launch_kwaves_tile(Params p, hipStream_t stream) {
  constexpr int MB = (AL + 3) / 4;
  constexpr int kPipe = kWaves * (MB + NB) * 4096, kSums = (MB > 1 ? 2 : 1) * kWaves * 4096 * NB;
  constexpr int kLds = kPipe > kSums ? kPipe : kSums;
  static_assert(kLds <= 160 * 1024, "LDS budget");
  p.tiles_m = (p.M + 8 * AL - 1) / (8 * AL);
  p.tiles_n = (p.N + 32 * NB - 1) / (32 * NB);
  auto kern = gemm_kernel_kwaves<P, AL, NB, kWaves>;
  static bool lds_limit_raised[kMaxDevices];
  if (raise_lds_limit<kLds>(kern, lds_limit_raised)) return -1;
  hipLaunchKernelGGL(kern, dim3((unsigned)kwaves_workgroups(KwavesForm{AL, NB, kWaves}, p.M, p.N)), dim3(64 * kWaves), kLds, stream, p);
  DQ_CHECK_HIP(hipGetLastError());
  return 0;
}

// What a call takes on each form (us): start + rounds x (round + K / 1000 x per_k), fitted over some hundred shapes a format
// (rows 2 to 500, N 1500 to 28500, K 1024 to 14300; mean error 5 to 9 %), where the form that they pick is 0.3 to 0.7 % slower in
// the mean than the best of the five.  Two workgroups of four waves share a CU, so their rounds of 256 run into each other;
// rounds of eight waves are counted whole.
struct KwavesCost {
  double start, round, per_k;
  bool smooth;
};
typedef KwavesCost KwavesCosts[kKwavesFormCount];

struct KwavesPick {
  int form;
  double us;
};
// What reading A takes (us) where no L2 holds it: once for every set of weight rows of an XCD, less the sets that run side by side,
// at 0.9 TB/s an XCD.
inline double kwaves_reread(const KwavesForm& f, int M, int N, size_t a_bytes) {
  const long passes = ((long)M + 8 * f.al - 1) / (8 * f.al), sets = (((long)N + 32 * f.nb - 1) / (32 * f.nb) + 7) / 8;
  const long beside = std::max(1L, (f.waves == 8 ? 32 : 64) / passes);
  return (double)a_bytes * (double)((sets + beside - 1) / beside) / 0.9e6;
}

// a_bytes: of the activations, where the estimate is to know that beyond 4 MB they do not stay in an L2.  The costs, fitted to 600 rows,
// do not (2100 shapes of int8 x 2-bit with more, calls by the ratio of reading A to their estimate: 1.0 of it to 0.75, 1.2 to 1, 1.4
// beyond; M = 776, N = 1136, K = 13056 51 us on sets of 32, 33 on 64); 0: as fitted.
inline KwavesPick kwaves_pick(const KwavesCosts& costs, int M, int N, int K, size_t a_bytes = 0) {
  KwavesPick best{-1, 1e30};
  for (int i = 0; i < kKwavesFormCount; ++i) {
    if (i == 0 && M > 16) continue;  // passes of 16 rows are never the best
    const long wgs = kwaves_workgroups(kKwavesForms[i], M, N);
    const double whole = (double)((wgs + 255) / 256);
    const double rounds = costs[i].smooth ? (wgs <= 256 ? 1.0 : 0.5 * ((double)wgs / 256.0 + whole)) : whole;
    double us = costs[i].start + rounds * (costs[i].round + costs[i].per_k * K * 1e-3);
    if (a_bytes > 4000000u) us = std::max(us, 0.5 * us + 0.8 * kwaves_reread(kKwavesForms[i], M, N, a_bytes));
    if (us < best.us) best = {i, us};
  }
  return best;
}

// What a call takes of its estimate, which counts K smoothly, while the waves walk whole chunks (128 bytes of a row of B, chunk_k of
// K): where those share out evenly less (int8 x 2-bit, 9000 shapes: 0.85 of it, 0.92 where the waves walk a fifth more than K, 1.0
// from a half more on).
inline double kwaves_even(const KwavesPick& pick, int K, int chunk_k) {
  const int waves = kKwavesForms[pick.form].waves, each = ((K + chunk_k - 1) / chunk_k + waves - 1) / waves;
  return std::min(1.0, 0.55 + 0.3 * each * waves * chunk_k / K);
}

// The share of a neighbour's estimate that this kernel's has to stay below.  Every set of weight rows reads all of A again: beyond a
// thousand rows and 8 MiB of it the L2s no longer serve that, which the costs, fitted to 600 rows, do not know (int8, 159 and 151
// shapes: 0.64 to 0.69 of the neighbour's time where the estimates' ratio is below 0.7, 1.0 to 1.15 of it above, up to 1.6; M = 3859,
// N = 256, K = 22272 60 us on the tiles of int8 x int4 and 98 here).  int8 x 2-bit, whose tiles' estimate is high there, counts the reads.
inline double kwaves_margin(double margin, int M, size_t a_bytes) { return M > 1000 && a_bytes > (8u << 20) ? 0.7 * margin : margin; }

template <class P>
int launch_kwaves(const Params& p, int form, hipStream_t stream) {
  static_assert(sizeof(kKwavesForms) / sizeof(kKwavesForms[0]) == 5, "one case a form");
  switch (form) {
    case 0: return launch_kwaves_tile<P, 2, 1, 8>(p, stream);
    case 1: return launch_kwaves_tile<P, 4, 1, 8>(p, stream);
    case 2: return launch_kwaves_tile<P, 4, 2, 4>(p, stream);
    case 3: return launch_kwaves_tile<P, 6, 2, 4>(p, stream);
    default: return launch_kwaves_tile<P, 8, 2, 4>(p, stream);
  }
}

}  // namespace gemm
}  // namespace dq
