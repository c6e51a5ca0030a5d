// Linear layers on few rows (M <= 64: one token of each of a few sequences),
// bf16 or int8 weights: y[m,n] = act(scale[n] sum_k x[m,k] w[n,k] + bias[n]).
//
// Bound: reading the weights once.  The tiles of gemm_core.hpp pad 8 rows to
// 128, move the weights through LDS and need a second launch to add their K
// slices.  Here a workgroup owns 16 NB output columns and all of K: its waves
// take a slice of K each, read the weights straight from memory in the layout
// of v_mfma_f32_16x16x32_bf16's A operand (lane (r, g): 16 consecutive k's of
// weight row r; a row's four lanes are 64 or 128 bytes together), and meet in
// LDS, in slice order.  Each weight is read by one lane of the chip, so LDS
// staging would only add a copy; x (the B operand) is small and comes through
// L2 in whole lines and a tile in the wave's own LDS (read straight into the
// operand's layout, 16 rows of 32 bytes a time, it took as long as the weights).
// Loads run one group of chunks ahead of the MFMAs.
#pragma once

#include "mfma.hpp"

namespace teeny {

// XR: rows of x, in MB blocks of 16 columns of the MFMA (columns past XR hold
// nothing and are not stored); NB: 16-row blocks of weights per wave; KW waves;
// U chunks of 64 k's in a load group.
template <bool INT8B, int XR, int NB, int KW, int U>
__global__ __launch_bounds__(64 * KW) void gemm_skinny(GemmParams p) {
  constexpr int MB = (XR + 15) / 16;
  constexpr int WV = INT8B ? 1 : 2;      // 16-byte weight vectors per lane and chunk
  constexpr int LX = 64 * U + 8;         // row stride of the x tile: no bank conflicts over 16 rows
  constexpr int NX = XR * 8 * U / 64;    // 16-byte x vectors per lane and group
  constexpr int LD = 16 * MB + 1;
  constexpr int XT = 16 * MB * LX / 2, RED = 16 * NB * LD;  // 4-byte words
  static_assert(XR * 8 * U % 64 == 0, "whole rounds of x loads");
  __shared__ __attribute__((aligned(16))) float lds[KW * (XT > RED ? XT : RED)];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * NB;
  const int chunks = p.K / 64 + (p.K % 64 != 0), per = (chunks + KW - 1) / KW;
  const int cb = min(chunks, w * per), ce = min(chunks, cb + per);
  bf16 *xt = reinterpret_cast<bf16 *>(lds + w * XT);
  // k's of lane group g in a chunk: 16 g .. 16 g + 15 (one 16-byte vector of
  // int8), or 8 g and 32 + 8 g (two of bf16)
  constexpr int KG = INT8B ? 16 : 8;
  using W = std::conditional_t<INT8B, int8_t, bf16>;
  const W *wrow[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
    wrow[i] = static_cast<const W *>(p.B) + static_cast<int64_t>(min(n0 + 16 * i + r, p.N - 1)) * p.ldb + KG * g;

  f32x4 acc[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  struct Group {
    u32x4 w[U][NB][WV], x[NX];
  };
  const u32x4 none = {0u, 0u, 0u, 0u};
  // chunks c .. c + U - 1; WHOLE: all of them exist and end by K.  Otherwise
  // what lies past K or the wave's slice reads as zero (K % 16 == 0: a vector
  // is inside or outside as a whole); its load goes to the row's start.  K may
  // be 2^31 - 16 and the last chunks then end past 2^31: compared unsigned.
  auto load = [&](auto whole_, Group &q, int c) __attribute__((always_inline)) {
    constexpr bool WHOLE = decltype(whole_)::value;
    const uint32_t k_end = min(64u * ce, static_cast<uint32_t>(p.K));
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int v = 0; v < WV; ++v) {
          const bool in = WHOLE || 64u * (c + u) + 32 * v + KG * g < k_end;
          q.w[u][i][v] = *reinterpret_cast<const u32x4 *>(wrow[i] + (in ? 64 * (c + u) + 32 * v : -KG * g));
          if (!in) q.w[u][i][v] = none;
        }
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int t = 64 * i + lane, col = 8 * (t % (8 * U));
      const bool in = WHOLE || 64u * c + col < k_end;
      const int64_t row = min(t / (8 * U), p.M - 1);
      q.x[i] = *reinterpret_cast<const u32x4 *>(p.A + row * p.lda + (in ? 64 * c + col : 0));
      if (!in) q.x[i] = none;
    }
  };
  auto multiply = [&](const Group &q) __attribute__((always_inline)) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int t = 64 * i + lane;
      *reinterpret_cast<u32x4 *>(xt + t / (8 * U) * LX + 8 * (t % (8 * U))) = q.x[i];
    }
    // the wave's lanes read what its other lanes wrote
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        bf16x8 x[MB];
#pragma unroll
        for (int j = 0; j < MB; ++j)
          x[j] = *reinterpret_cast<const bf16x8 *>(xt + (16 * j + r) * LX + 64 * u + KG * g + (INT8B ? 8 : 32) * v);
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          bf16x8 a;
          if constexpr (INT8B) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const uint32_t word = q.w[u][i][0][2 * v + (j >> 1)] >> (16 * (j & 1));
              const bf16x2 pr = cvt_pk_bf16(static_cast<float>(static_cast<int8_t>(word & 0xffu)),
                                            static_cast<float>(static_cast<int8_t>((word >> 8) & 0xffu)));
              a[2 * j] = pr[0];
              a[2 * j + 1] = pr[1];
            }
          } else {
            a = __builtin_bit_cast(bf16x8, q.w[u][i][WV == 2 ? v : 0]);
          }
#pragma unroll
          for (int j = 0; j < MB; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, x[j], acc[i][j], 0, 0, 0);
        }
      }
  };
  // whole groups, the next one's loads ahead of this one's products
  const int k_whole = min(ce, p.K / 64);  // chunks below it end by K
  Group a, b;
  int c = cb;
  if (c + U <= k_whole) {
    load(std::true_type{}, a, c);
    c += U;
    while (c + 2 * U <= k_whole) {
      load(std::true_type{}, b, c);
      multiply(a);
      load(std::true_type{}, a, c + U);
      multiply(b);
      c += 2 * U;
    }
    if (c + U <= k_whole) {
      load(std::true_type{}, b, c);
      multiply(a);
      multiply(b);
      c += U;
    } else {
      multiply(a);
    }
  }
  if (c < ce) {  // fewer than U whole chunks and the one that K ends in
    load(std::false_type{}, a, c);
    multiply(a);
  }
  __syncthreads();

  // D: lane (r, g) holds column (x row) r, weight rows 4 g .. 4 g + 3
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) lds[w * RED + (16 * i + 4 * g + e) * LD + 16 * j + r] = acc[i][j][e];
  __syncthreads();
  for (int t = threadIdx.x; t < 16 * NB * XR; t += 64 * KW) {
    const int m = t / (16 * NB), n = t % (16 * NB);
    if (m >= p.M || n0 + n >= p.N) continue;
    float v = lds[n * LD + m];
#pragma unroll
    for (int i = 1; i < KW; ++i) v += lds[i * RED + n * LD + m];
    if (p.scale != nullptr) v *= p.scale[n0 + n];
    if (p.bias != nullptr) v += p.bias[n0 + n];
    if (p.bias_bf16 != nullptr) v += static_cast<float>(p.bias_bf16[n0 + n]);
    p.C[m * p.ldc + n0 + n] = static_cast<bf16>(apply_act_rt(v, p.act));
  }
}

// Weight blocks per wave.  More of them read x less often, which counts from
// 17 rows on, but leave fewer workgroups: the most that still give 160 of them
// (us, int8, 32 rows: N x K = 11008 x 4096 with 1 / 2 / 4 blocks 23.8 / 21.9 /
// 19.2, 4096 x 11008 20.0 / 24.9 / 38.9).
inline int gemm_skinny_nb(int64_t M, int64_t N) { return M <= 16 || N < 16 * 2 * 160 ? 1 : N < 16 * 4 * 160 ? 2 : 4; }

// Whether this kernel is the better one: plain 16-byte aligned rows, K a
// multiple of 16, up to 64 rows.  us against the tiles and their K slices,
// int8: 8 rows 4096 -> 11008 26.5 / 14.3, 11008 -> 4096 45.6 / 15.0; 64 rows
// 29.3 / 24.1 and 46.5 / 29.6.  bf16: 8 rows 27.1 / 21.3 and 47.1 / 21.7; 64
// rows 31.1 / 33.0 and 48.2 / 37.3, so wide bf16 outputs stay there past 32
// rows.  So do narrow ones (fewer than 64 workgroups here) whose K the tiles
// split.  Weights rotated through 600 MB.
inline bool gemm_skinny_ok(bool int8, int64_t M, int64_t N, int64_t K) {
  if (K % 16 != 0 || M > 64) return false;
  // 2^32 threads in a grid (more of them wrap): the tiles want 4 a column, not 32
  if (cdiv(N, 16 * gemm_skinny_nb(M, N)) >= (int64_t{1} << 32) / 512) return false;
  return M <= 32 || ((N >= 16 * 64 || K < 2048) && (int8 || gemm_skinny_nb(M, N) < 4));
}

template <bool INT8B> inline void launch_gemm_skinny(GemmParams p, int act, hipStream_t s) {
  p.act = act;
  const int nb = gemm_skinny_nb(p.M, p.N);
#define TEENY_SKINNY(XR, NB, U)                                                                         \
  hipLaunchKernelGGL((gemm_skinny<INT8B, XR, NB, 8, U>), dim3(static_cast<unsigned>(cdiv(p.N, 16 * NB))), \
                     dim3(512), 0, s, p)
  if (p.M <= 2) TEENY_SKINNY(2, 1, 4);
  else if (p.M <= 8) TEENY_SKINNY(8, 1, 4);
  else if (p.M <= 16) TEENY_SKINNY(16, 1, 2);
  else if (p.M <= 32 && nb == 1) TEENY_SKINNY(32, 1, 2);
  else if (p.M <= 32 && nb == 2) TEENY_SKINNY(32, 2, 2);
  else if (p.M <= 32) TEENY_SKINNY(32, 4, 1);
  else if (nb == 1) TEENY_SKINNY(64, 1, 1);
  else if (nb == 2) TEENY_SKINNY(64, 2, 1);
  else if constexpr (INT8B) TEENY_SKINNY(64, 4, 1);  // bf16: gemm_skinny_ok
#undef TEENY_SKINNY
}

}  // namespace teeny
