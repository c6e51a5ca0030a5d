// Attention forward for few query rows, bf16 at head_dim 64 and 128 (one token
// at a time, a few draft tokens, short prompts, few heads): the keys of a head
// are shared out over waves and workgroups.
//
// Bound: reading K and V once.  fa_fwd_bf16 gives each query head a workgroup
// of 128 query rows, so with one query it multiplies mostly padding, reads a
// K/V head once per query head that shares it, and runs as many workgroups
// as there are heads.  Here the query rows that share a K/V head (its query
// heads times their queries, consecutive in memory) are packed into column
// blocks of 32 (causal and more than 32 queries: a head's rows start a new
// block, whose keys then end with its own last query's, so that a row meets
// no masked key past the 32-key tile of its block's last row, whose V may
// hold an infinity or NaN); a workgroup of four waves takes one block and a range of the
// keys, each wave every fourth 32-key tile of it, and the workgroups of a
// block meet through the stream's workspace (fp32 partial outputs with their
// max and sum, combined by a second small kernel in range order).
// A wave works alone, with no barrier in its loop: S^T = K Q^T takes K's
// fragments straight from memory to registers (each is used once, so LDS
// would only add a copy), V's tile goes through the wave's own LDS for the
// transposing read.  Both are refilled as soon as they are used, so a wave
// has up to 16 KiB in flight, 128 KiB per CU, which covers the latency at
// the full HBM rate.  Rounding points are fa_fwd_bf16's: probabilities to
// bf16, everything else fp32.
#pragma once

#include "mfma.hpp"

namespace teeny {

struct AttnSplitArgs {
  const bf16 *Q, *K, *V;
  bf16 *O;
  float *L;
  float *part;        // [unit][range][row][D] fp32, then [unit][range][row][2]; null: one range
  int64_t ml_off;     // offset of the second array in floats
  int rows;           // query rows of a run that blocks are cut from: a K/V head's, or one query head's
  int kv_runs;        // runs per K/V head
  int nq;             // queries per query head
  int blocks;         // column blocks per run
  int nk, range;      // keys, keys per range (a multiple of 32)
  float scale_log2;
};

template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void fa_split_bf16(AttnSplitArgs p) {
  constexpr int CPR = D / 8, RPB = 128 / D, NS = D / 16, ND = D / 32, NV = 32 * CPR / 64;
  constexpr int RED = D * 33;  // a wave's partial output [D][33]
  __shared__ __attribute__((aligned(16))) float red[4][RED];
  __shared__ float ml[2][4][32];
  static_assert(RED * 4 >= 32 * D * 2, "the V tile shares the reduction's space");
  auto fv = [](int row) { return (4 * (row / RPB)) & (CPR - 1) & ~3; };
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 31, g = lane >> 5;
  const uint32_t unit = blockIdx.y;  // (run, column block)
  const uint32_t run = unit / static_cast<uint32_t>(p.blocks), hk = run / static_cast<uint32_t>(p.kv_runs);
  const int c0 = static_cast<int>(unit - run * p.blocks) * 32, ncol = min(32, p.rows - c0);
  const int64_t row0 = static_cast<int64_t>(run) * p.rows + c0, key0 = static_cast<int64_t>(hk) * p.nk;
  const bf16 *Kb = p.K + key0 * D, *Vb = p.V + key0 * D;
  // causal: the row's query sees the keys up to its own index, the block's rows those up to their last one's
  // (of several heads in a block, which have at most 32 queries, up to the heads' last)
  const int qi = CAUSAL ? (c0 + min(c, ncol - 1)) % p.nq : 0;
  int k_end = p.nk;
  if constexpr (CAUSAL) k_end = min(p.nk, c0 % p.nq + ncol > p.nq ? p.nq : c0 % p.nq + ncol);
  const int kb = blockIdx.x * p.range, ke = min(k_end, kb + p.range);
  bf16 *vt = reinterpret_cast<bf16 *>(red[w]);

  const float sc = fmaxf(fabsf(p.scale_log2), 1.17549435e-38f);  // as fa_fwd_bf16: the sign goes to Q
  const uint32_t qsign = p.scale_log2 < 0.0f ? 0x80008000u : 0u;
  bf16x8 qf[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    u32x4 raw = *reinterpret_cast<const u32x4 *>(p.Q + (row0 + min(c, ncol - 1)) * D + 16 * s + 8 * g);
    raw ^= qsign;
    __builtin_memcpy(&qf[s], &raw, 16);
  }
  f32x16 acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) acc[d] = zero16();
  float m_run = -INFINITY, l_run = 0.0f;

  // the transposing read of V (see fa_fwd_bf16)
  const int hh = lane >> 4, m16 = lane & 15, v_row = 4 * g + (m16 >> 2);
  const int vofs = v_row * D + ((fv(v_row) | (2 * (hh & 1) + ((m16 & 3) >> 1))) << 3) + (m16 & 1) * 4;

  u32x4 kr[NS], vr[NV];
  auto load_k = [&](int k0) {
    const bf16 *row = Kb + static_cast<int64_t>(min(k0 + c, p.nk - 1)) * D + 8 * g;
#pragma unroll
    for (int s = 0; s < NS; ++s) kr[s] = *reinterpret_cast<const u32x4 *>(row + 16 * s);
  };
  auto load_v = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int t = 64 * i + lane;
      const int64_t row = min(k0 + t / CPR, p.nk - 1);
      vr[i] = *reinterpret_cast<const u32x4 *>(Vb + row * D + 8 * (t % CPR));
    }
  };
  int k0 = kb + 32 * w;
  if (k0 < ke) {
    load_k(k0);
    load_v(k0);
  }
  for (; k0 < ke; k0 += 128) {
    f32x16 s = zero16();
#pragma unroll
    for (int i = 0; i < NS; ++i) s = mfma32x32x16(__builtin_bit_cast(bf16x8, kr[i]), qf[i], s);
    const bool more = k0 + 128 < ke, edge = k0 + 32 > p.nk;
    const bool masks = edge || (CAUSAL && __any(k0 + 31 > qi));
    if (more) load_k(k0 + 128);
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      if (masks && (k0 + mfma32_row(v, g) >= p.nk || (CAUSAL && k0 + mfma32_row(v, g) > qi))) s[v] = -INFINITY;
      mx = __builtin_elementwise_maximum(mx, s[v]);
    }
    mx = __builtin_elementwise_maximum(mx, __shfl_xor(mx, 32, 64)) * sc;
    if (__any(mx > m_run + 8.0f)) {  // rescaled rarely, as in fa_fwd_bf16: p <= 2^8
      const float m_new = fmaxf(m_run, mx);
      const float alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.0f : m_new));
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < ND; ++d) acc[d] *= alpha;
      m_run = m_new;
    }
    const float neg_m = m_run == -INFINITY ? 0.0f : -m_run;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      s[v] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[v], sc, neg_m));
      l_run += s[v];
    }
    // rows past nk are zeros, so that a zero probability meets no stray infinity
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int t = 64 * i + lane, r = t / CPR;
      u32x4 v = vr[i];
      if (edge && k0 + r >= p.nk) v = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4 *>(vt + r * D + (((t % CPR) ^ fv(r)) << 3)) = v;
    }
    if (more) load_v(k0 + 128);
    // the wave's lanes read what its other lanes wrote
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      bf16x8 pb;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bf16x2 pr = cvt_pk_bf16(s[8 * tt + 2 * j], s[8 * tt + 2 * j + 1]);
        pb[2 * j] = pr[0];
        pb[2 * j + 1] = pr[1];
      }
#pragma unroll
      for (int d = 0; d < ND; ++d) {
        const bf16 *vp = vt + 16 * tt * D + (vofs ^ (d << 5));
        const bf16x4 lo = ds_read_tr16(vp), hi = ds_read_tr16(vp + 8 * D);
        acc[d] = mfma32x32x16(cat8(lo, hi), pb, acc[d]);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  l_run += __shfl_xor(l_run, 32, 64);

  // the four waves' parts: a common max, then the sum of their outputs
  if (g == 0) {
    ml[0][w][c] = m_run;
    ml[1][w][c] = l_run;
  }
  __syncthreads();
  float m = ml[0][0][c], l = 0.0f;
#pragma unroll
  for (int i = 1; i < 4; ++i) m = fmaxf(m, ml[0][i][c]);
  const float ref = m == -INFINITY ? 0.0f : m;
#pragma unroll
  for (int i = 0; i < 4; ++i) l += ml[1][i][c] * __builtin_amdgcn_exp2f(ml[0][i][c] - ref);
  const bool whole = p.part == nullptr;
  const float mul = __builtin_amdgcn_exp2f(m_run - ref) * (whole ? 1.0f / l : 1.0f);
  if (c < ncol) {
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int v = 0; v < 16; ++v) red[w][(32 * d + mfma32_row(v, g)) * 33 + c] = acc[d][v] * mul;
  }
  __syncthreads();
  const int64_t slot = (static_cast<int64_t>(unit) * gridDim.x + blockIdx.x) * 32;  // part rows of this (unit, range)
  for (int i = threadIdx.x; i < ncol * (D / 4); i += 256) {
    const int r = i / (D / 4), d = 4 * (i % (D / 4));
    f32x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int at = (d + j) * 33 + r;
      o[j] = (red[0][at] + red[1][at]) + (red[2][at] + red[3][at]);
    }
    if (whole) {
      bf16x4 o4;
#pragma unroll
      for (int j = 0; j < 4; ++j) o4[j] = static_cast<bf16>(o[j]);
      *reinterpret_cast<bf16x4 *>(p.O + (row0 + r) * D + d) = o4;
    } else {
      *reinterpret_cast<f32x4 *>(p.part + (slot + r) * D + d) = o;
    }
  }
  if (w == 0 && g == 0 && c < ncol) {
    if (!whole) {
      p.part[p.ml_off + (slot + c) * 2] = m;
      p.part[p.ml_off + (slot + c) * 2 + 1] = l;
    } else if (p.L != nullptr) {
      p.L[row0 + c] = (m + log2f(l)) * 0.6931471805599453f;
    }
  }
}

// One wave per query row: the ranges' parts, in range order.
template <int D>
__global__ __launch_bounds__(256) void fa_split_combine(AttnSplitArgs p, int ranges, int64_t total) {
  constexpr int V = D / 64;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= total) return;
  const int64_t run = row / p.rows;
  const int r = static_cast<int>(row - run * p.rows);
  const int64_t slot = (run * p.blocks + r / 32) * ranges * 32 + r % 32;
  const float *ml = p.part + p.ml_off;
  float m = -INFINITY;
  for (int i = 0; i < ranges; ++i) m = fmaxf(m, ml[(slot + 32 * i) * 2]);
  const float ref = m == -INFINITY ? 0.0f : m;
  float l = 0.0f, o[V] = {};
  for (int i = 0; i < ranges; ++i) {
    const float f = __builtin_amdgcn_exp2f(ml[(slot + 32 * i) * 2] - ref);
    l += ml[(slot + 32 * i) * 2 + 1] * f;
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] = __builtin_fmaf(p.part[(slot + 32 * i) * D + lane * V + j], f, o[j]);
  }
  const float inv = 1.0f / l;
#pragma unroll
  for (int j = 0; j < V; ++j) p.O[row * D + lane * V + j] = static_cast<bf16>(o[j] * inv);
  if (p.L != nullptr && lane == 0) p.L[row] = (m + log2f(l)) * 0.6931471805599453f;
}

// Whether this path is the better one, and into how many ranges it cuts the
// keys.  fa_fwd_bf16 is the faster kernel on a full chip; its workgroups are
// four column blocks each, so it wants four times the blocks to fill it.
// Measured in us (heads x queries x keys x head_dim; fa_fwd_bf16 / here): 256
// blocks, 16 x 512 x 512 x 64 causal 11.9 / 7.7, 4 x 2048 x 2048 x 128 causal
// 41.0 / 26.4, 8 x 1024 x 1024 x 128 22.3 / 16.6; 512 blocks, not causal 16 x
// 1024 x 1024 x 128 23.4 / 27.8, 4 x 4096 x 4096 x 128 71.6 / 81.1.  Causal its
// longest block sets the time until every CU has several to run: at 512 blocks
// head_dim 64 still gains here, 16 x 1024 x 1024 18.4 / 15.5, 32 x 512 x 512
// 12.0 / 10.2, 8 x 2048 x 2048 30.8 / 24.6, while 128 does not, 16 x 1024 x 1024
// 25.2 / 27.4, 32 x 512 x 512 16.5 / 17.7, 8 x 2048 x 2048 41.1 / 44.5;
// 1024 blocks, 64 x 512 x 512 x 128 16.6 / 32.0.  At up to 32 queries most of
// fa_fwd_bf16's rows are padding: 32 heads sharing 8 K/V heads, one query, batch
// x keys 1 x 16384 262 / 31, 32 x 1000 57 / 23, 16 x 4000 106 / 52 (5 TB/s).  On
// a full chip that counts where packing leaves fewer blocks than heads (heads in
// groups of 4 or 8; queries x keys x head_dim): 32 x 2048 x 128, as many blocks
// as heads, 256 of them 38 / 41, 512 55 / 79, 4096 1.19 times as long; 20 x 2048 x 128, 5
// blocks to 8 heads, 320 54 / 61, 640 0.93; half as many blocks or fewer 0.16 to
// 0.77 at any size.  head_dim 64, 32 x 2048, as many blocks as heads: 512 35 /
// 40, 2048 1.09, 4096 0.9; fewer blocks than heads, or causal and so one tile of
// keys, 0.1 to 1.07.  Heads that share no K/V gain (0.94 and 0.89 on average)
// but for one tile of keys per wave at 128, 512 x 32 x 64 6.9 / 8.5.  With so
// few keys at head_dim 128 also a chip that is not full waits for this path's
// longer way to its first product and its merge: 16 x 32 x 64 5.0 / 5.9, 33 x
// 128 5.6 / 6.2, but 100 x 128 0.94 and with 4 rows 0.96.  Ranges cost a second
// launch and pay from about 512 keys each: 8 x 64 x 2048 25.3 -> 15.1, 8 x 128 x
// 4096 44.3 -> 19.0, but 8 x 128 x 512 11.0 -> 12.3 with two.
struct AttnSplitPlan {
  bool use = false;
  int64_t units = 0;
  int rows = 0, kv_runs = 1, blocks = 0, ranges = 1, range = 0;
  size_t bytes = 0;  // workspace of the ranges
};

// BH query heads of nq rows, group of them to a K/V head.  Causal, no query
// sees a key past the last one's: ranges that shared those out too were mostly
// empty workgroups (8 heads of 64 queries x 16384 keys x 128 29 -> 6 us).
inline AttnSplitPlan attn_split_plan(int64_t BH, int64_t group, int64_t nq, int64_t nk, int64_t D, bool causal,
                                     size_t scratch) {
  AttnSplitPlan pl;
  if (causal) nk = std::min(nk, nq);
  const int64_t kv_runs = causal && nq > 32 ? group : 1, rows = group / kv_runs * nq;
  const int64_t cus = device_cu_count(), blocks = cdiv(rows, 32), units = BH / group * kv_runs * blocks;
  const int64_t room = causal && nq > 128 && D == 64 ? 2 * cus : D == 128 && !causal && nq <= 64 ? cus - 1 : cus;
  if (units > room) {
    const bool packed = D == 64 ? units < BH || units > 8 * cus || nk <= 32
                                : 2 * units <= BH || (4 * units <= 3 * BH && units > 3 * cus);
    if (nq > 32 || (group > 1 ? !packed : D == 128 && nq > 16 && nk <= 64)) return pl;
  }
  if (D == 128 && !causal && nk <= 128 && nq <= 64 && group * nq > 8 && BH <= cus) return pl;
  pl.use = true;
  pl.units = units;
  pl.rows = static_cast<int>(rows);
  pl.kv_runs = static_cast<int>(kv_runs);
  pl.blocks = static_cast<int>(blocks);
  int64_t ranges = units > cus / 2 ? 1 : std::max<int64_t>(1, std::min(2 * cus / units, nk / 512));
  auto size = [&](int64_t n) { return n > 1 ? static_cast<size_t>(units) * n * 32 * (D + 2) * 4 : 0; };
  if (size(ranges) > scratch) ranges = 1;
  pl.range = static_cast<int>(cdiv(cdiv(nk, ranges), 32) * 32);
  pl.ranges = static_cast<int>(cdiv(nk, pl.range));
  pl.bytes = size(pl.ranges);
  return pl;
}

template <int D, bool CAUSAL>
inline void attn_split_launch(const AttnSplitPlan &pl, AttnSplitArgs p, hipStream_t s) {
  p.rows = pl.rows;
  p.kv_runs = pl.kv_runs;
  p.blocks = pl.blocks;
  p.range = pl.range;
  p.ml_off = pl.units * pl.ranges * 32 * D;
  if (pl.ranges == 1) p.part = nullptr;
  hipLaunchKernelGGL((fa_split_bf16<D, CAUSAL>), dim3(pl.ranges, static_cast<unsigned>(pl.units)), dim3(256), 0, s, p);
  if (pl.ranges > 1) {
    const int64_t total = pl.units / pl.blocks * p.rows;
    hipLaunchKernelGGL(fa_split_combine<D>, dim3(static_cast<unsigned>(cdiv(total, 4))), dim3(256), 0, s, p, pl.ranges,
                       total);
  }
}

}  // namespace teeny
