// Attention forward and backward with fp32 products on the fp32 matrix cores:
// fp32 tensors at head_dim 16 .. 128, and bf16 tensors where the bf16 MFMA
// kernels do not apply (head_dim 16 and 32; dk/dv without a workspace or with
// unaligned tensors), widened on load.  fp32 everywhere between.
//
// Bound: v_mfma_f32_32x32x2_f32 (157 TFLOP/s; 64 cycles for each 32 x 32 x 2).
// At that rate a wave needs little from LDS (one 4-byte read per lane and
// MFMA for the transposed operand, a quarter of a 16-byte one for the other)
// and 32 rows of operands give 16 FLOP per byte from L2, so every wave works
// alone: it owns 32 columns (queries in the forward and dq, keys in dk/dv)
// with their operands and accumulators in registers, and walks tiles of 32
// rows of the other side through LDS tiles of its own, with no barrier in the
// loop.  Tiles go global -> registers -> LDS: one operand's next tile is in
// flight while the other's product runs.  As in the bf16 kernels the scores
// are computed with the wave's columns as the MFMA's columns, so that softmax
// rows are in-lane and P (and dS) feed the next product from the registers
// they were computed in: register r of lane (c, h) is row 8 (r / 4) + 4 h +
// r % 4 of column c, which is also the k that the next product's step r
// gives that lane.
//
// Small grids give each block of 32 columns to a workgroup whose waves share
// out the tiles and merge in LDS: eight waves (two per SIMD, head_dim up to
// 64) while the blocks do not outnumber the CUs, four below 2048 blocks;
// otherwise the four waves of a workgroup take a block each.  Results do not
// depend on timing (no atomics).
//
// Measured, 16 heads of 500 x 500 x 64 fp32, forward + dq + dk/dv: 2987 us
// with one wave per row (152 + 288 + 2504) -> 69 us (18 + 24 + 32 traced), 67
// TFLOP/s of the nine products executed (256 blocks of 32 columns, one
// workgroup per CU: 2048 waves, two per SIMD, with two 32 x 32 tiles each).
// dk/dv holds two operands and two accumulators: at head_dim 64 all of its 256
// registers with 39 to 54 spilled (84 to 104 bytes a lane), at 128 28 to 37
// beside the accumulation registers, reloaded in the tile loop.
//
// A product with a masked pair is p = 0 times a row that the query may not
// see; if such a row holds an infinity or NaN the tile is redone pair by pair
// (masked_outer), so that it reaches only the queries that see it.
#pragma once

#include <algorithm>

#include "mfma.hpp"

namespace teeny {

typedef float fa_f32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef bf16 fa_bf16x4u __attribute__((ext_vector_type(4), aligned(2)));
template <typename T> struct FaVec4;
template <> struct FaVec4<float> {
  typedef fa_f32x4u type;
  static __device__ __forceinline__ f32x4 wide(fa_f32x4u v) { return v; }
};
template <> struct FaVec4<bf16> {
  typedef fa_bf16x4u type;
  static __device__ __forceinline__ f32x4 wide(fa_bf16x4u v) {
    return f32x4{to_f32(v[0]), to_f32(v[1]), to_f32(v[2]), to_f32(v[3])};
  }
};
template <typename T> __device__ __forceinline__ f32x4 fa_load4(const T *p) {
  return FaVec4<T>::wide(*reinterpret_cast<const typename FaVec4<T>::type *>(p));
}

// Orders this wave's LDS writes before its later reads, across lanes.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// exp(d) to about an ulp: v_exp_f32 of the rounded d log2(e), corrected to
// first order by what that rounding left out.
__device__ __forceinline__ float exp_near(float d) {
  constexpr float kL = 1.4426950408889634f, kLlo = 1.9259629911266175e-8f, kLn2 = 0.6931471805599453f;
  const float t = d * kL;
  const float e = __builtin_fmaf(d, kLlo, __builtin_fmaf(d, kL, -t));
  const float p = __builtin_amdgcn_exp2f(t);
  return fabsf(t) < 127.0f ? __builtin_fmaf(p, e * kLn2, p) : p;
}

__device__ __forceinline__ float other_half(float v) { return __shfl_xor(v, 32, 64); }

// Row and column indexes are unsigned: a count may be 2^31 - 1 and the last
// block of 32 then ends past it.
//
// 32 rows of [n, D] on their way from memory to a wave's LDS tile [32][LD].
// LD = D + 8 keeps both reads free of bank conflicts: 16 bytes of 8 rows, and
// one word of two rows 4 apart.
template <typename T, int D> struct FaTile {
  static constexpr int LD = D + 8, CH = D / 4, NV = D / 8;
  static constexpr int FLOATS = 32 * LD;
  typename FaVec4<T>::type r[NV];
  __device__ __forceinline__ void fetch(const T *base, uint32_t r0, uint32_t n, int lane) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int t = i * 64 + lane;
      const int64_t row = min(r0 + static_cast<uint32_t>(t / CH), n - 1);
      r[i] = *reinterpret_cast<const typename FaVec4<T>::type *>(base + row * D + 4 * (t % CH));
    }
  }
  // Rows past n are zeros.  Whether any value is an infinity or NaN, if asked.
  template <bool CHECK = false>
  __device__ __forceinline__ bool store(float *lds, uint32_t r0, uint32_t n, int lane) const {
    bool odd = false;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int t = i * 64 + lane;
      f32x4 v = FaVec4<T>::wide(r[i]);
      if (r0 + 32 > n && r0 + t / CH >= n) v = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if constexpr (CHECK) {
#pragma unroll
        for (int j = 0; j < 4; ++j) odd |= !(fabsf(v[j]) <= 3.402823466e38f);
      }
      *reinterpret_cast<f32x4 *>(lds + t / CH * LD + 4 * (t % CH)) = v;
    }
    return odd;
  }
};

// The wave's 32 columns as an MFMA operand: lane (c, h) has elements
// 8 j + 4 h .. + 3 of row c0 + c (the last row again past n).
template <typename T, int D>
__device__ __forceinline__ void fa_cols(f32x4 (&b)[D / 8], const T *base, uint32_t c0, uint32_t n, int c, int h) {
  const T *p = base + static_cast<int64_t>(min(c0 + c, n - 1)) * D + 4 * h;
#pragma unroll
  for (int j = 0; j < D / 8; ++j) b[j] = fa_load4(p + 8 * j);
}

// tile [32][D] times the columns: rows of the tile x columns.
template <int D>
__device__ __forceinline__ f32x16 fa_inner(const float *tile, const f32x4 (&b)[D / 8], int c, int h) {
  f32x16 s = zero16();
#pragma unroll
  for (int j = 0; j < D / 8; ++j) {
    const f32x4 a = *reinterpret_cast<const f32x4 *>(tile + c * (D + 8) + 8 * j + 4 * h);
#pragma unroll
    for (int i = 0; i < 4; ++i) s = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j][i], s, 0, 0, 0);
  }
  return s;
}

template <int D> struct FaAcc {
  static constexpr int ND = (D + 31) / 32;
  f32x16 a[ND];
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int d = 0; d < ND; ++d) a[d] = zero16();
  }
  // a[d][col] += sum over the tile's rows of tile[row][d] x[row][col]
  __device__ __forceinline__ void outer(const float *tile, const f32x16 &x, int c, int h) {
    const int cc = D < 32 ? min(c, D - 1) : c;  // rows d >= D are never stored
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float *row = tile + (8 * (r / 4) + 4 * h + r % 4) * (D + 8);
#pragma unroll
      for (int d = 0; d < ND; ++d)
        a[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(row[32 * d + cc], x[r], a[d], 0, 0, 0);
    }
  }
  // The same with the rows where seen(row) is false left out, not multiplied by zero.
  template <typename F>
  __device__ __forceinline__ void masked_outer(const float *tile, const f32x16 &x, int h, F seen) {
    for (int r = 0; r < 16; ++r) {
      float mine = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) mine = i == r ? x[i] : mine;
      const float their = other_half(mine);
      for (int hh = 0; hh < 2; ++hh) {
        const int row = 8 * (r / 4) + 4 * hh + r % 4;
        const float xv = hh == h ? mine : their;
        if (!seen(row)) continue;
#pragma unroll
        for (int d = 0; d < ND; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int dd = 32 * d + 8 * (i / 4) + 4 * h + i % 4;
            a[d][i] = __builtin_fmaf(tile[row * (D + 8) + min(dd, D - 1)], xv, a[d][i]);
          }
      }
    }
  }
  // to [D][33] floats, column fast
  __device__ __forceinline__ void put(float *red, float mul, int c, int h) const {
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int dd = 32 * d + 8 * (i / 4) + 4 * h + i % 4;
        if (D % 32 == 0 || dd < D) red[dd * 33 + c] = a[d][i] * mul;
      }
  }
};

// Writes rows c0 .. c0 + 31 (below n) of out [n, D] from the sum of `parts`
// [D][33] blocks `stride` floats apart; `step` threads, this one `t`.
template <typename T, int D, int PARTS>
__device__ __forceinline__ void fa_write(T *out, uint32_t c0, uint32_t n, const float *red, int stride, int t,
                                         int step) {
  for (int i = t; i < 32 * (D / 4); i += step) {
    const int row = i / (D / 4), d = 4 * (i % (D / 4));
    if (c0 + row >= n) continue;
    typename FaVec4<T>::type v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float s = red[(d + j) * 33 + row];
#pragma unroll
      for (int p = 1; p < PARTS; ++p) s += red[p * stride + (d + j) * 33 + row];
      v[j] = from_f32<T>(s);
    }
    *reinterpret_cast<typename FaVec4<T>::type *>(out + static_cast<int64_t>(c0 + row) * D + d) = v;
  }
}

// Waves of a workgroup: those that share a column block, or four blocks' own.
template <int SPLIT> constexpr int kFaWaves = SPLIT == 1 ? 4 : SPLIT;

// blocks of 32 columns: this wave's (column block, head), its share of the
// tiles, or false past the last block.  Grid (x, heads).
template <int SPLIT>
__device__ __forceinline__ bool fa_unit(int w, int blocks, int &blk, int64_t &head) {
  const int64_t total = static_cast<int64_t>(gridDim.x) * gridDim.y;
  int64_t id = static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
  if (total <= 0x7fffffff) id = xcd_remap(static_cast<int>(id), static_cast<int>(total));
  head = id / gridDim.x;
  const int x = static_cast<int>(id - head * gridDim.x);
  blk = SPLIT == 1 ? 4 * x + w : x;
  return blk < blocks;
}

template <typename T, int D, int SPLIT>
__global__ __launch_bounds__(64 * kFaWaves<SPLIT>, D <= 64 ? 2 : 1) void fa_fwd_f32(
    const T *__restrict__ Q, const T *__restrict__ K, const T *__restrict__ V, T *__restrict__ O,
    float *__restrict__ L, uint32_t nq, uint32_t nk, float scale, int causal, int kv_group, int nqb) {
  using Tile = FaTile<T, D>;
  __shared__ __attribute__((aligned(16))) float lds[kFaWaves<SPLIT>][2 * Tile::FLOATS];
  __shared__ float ml[2][kFaWaves<SPLIT>][32];
  // wave-uniform, so that the tile loop and its masks are scalar branches
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  int qb;
  int64_t bh;
  if (!fa_unit<SPLIT>(w, nqb, qb, bh)) return;
  if (causal) qb = nqb - 1 - qb;  // the longest first
  const uint32_t q0 = 32u * qb, qi = q0 + c;
  const T *Kb = K + (bh / kv_group) * nk * D, *Vb = V + (bh / kv_group) * nk * D;
  float *kt = lds[w], *vt = lds[w] + Tile::FLOATS;

  f32x4 q[D / 8];
  fa_cols<T, D>(q, Q + bh * nq * D, q0, nq, c, h);
  FaAcc<D> acc;
  acc.zero();
  float m = -INFINITY, l = 0.0f;  // l: this lane's keys only
  const uint32_t kend = causal ? min(nk, min(q0 + 32, nq)) : nk;
  const int tiles = static_cast<int>((kend + 31) / 32);
  int t = SPLIT == 1 ? 0 : w;
  Tile ts;
  if (t < tiles) {
    ts.fetch(Kb, 32 * t, nk, lane);
    ts.store(kt, 32 * t, nk, lane);
    wave_fence();
  }
  for (; t < tiles; t += SPLIT) {
    const uint32_t k0 = 32u * t;
    ts.fetch(Vb, k0, nk, lane);
    f32x16 s = fa_inner<D>(kt, q, c, h);
    const bool diag = causal && k0 + 31 > q0;
    const uint32_t last = causal ? min(kend - 1, qi) : kend - 1;  // last key that this lane's query sees
    float mx = m;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] *= scale;
    if (diag || k0 + 32 > kend) {
      asm volatile("" ::: "memory");  // a branch: whole tiles compare nothing
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = k0 + 8 * (r / 4) + 4 * h + r % 4 > last ? -INFINITY : s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, other_half(mx));
    const float ref = mx == -INFINITY ? 0.0f : mx;
    if (__any(mx > m)) {
      const float f = exp_near(m - ref);
      l *= f;
#pragma unroll
      for (int d = 0; d < FaAcc<D>::ND; ++d) acc.a[d] *= f;
      m = mx;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = exp_near(s[r] - ref);
      l += s[r];
    }
    const bool odd = diag ? ts.template store<true>(vt, k0, nk, lane) : ts.store(vt, k0, nk, lane);
    wave_fence();
    if (t + SPLIT < tiles) ts.fetch(Kb, k0 + 32 * SPLIT, nk, lane);
    if (diag && __any(odd))
      acc.masked_outer(vt, s, h, [&](int row) { return k0 + row <= last; });
    else
      acc.outer(vt, s, c, h);
    if (t + SPLIT < tiles) {
      ts.store(kt, k0 + 32 * SPLIT, nk, lane);
      wave_fence();
    }
  }
  l += other_half(l);

  float mul;
  T *Ob = O + bh * nq * D;
  if constexpr (SPLIT > 1) {
    if (h == 0) {
      ml[0][w][c] = m;
      ml[1][w][c] = l;
    }
    __syncthreads();
    float mx = ml[0][0][c], sum = 0.0f;
#pragma unroll
    for (int i = 1; i < SPLIT; ++i) mx = fmaxf(mx, ml[0][i][c]);
    const float ref = mx == -INFINITY ? 0.0f : mx;
#pragma unroll
    for (int i = 0; i < SPLIT; ++i) sum += ml[1][i][c] * exp_near(ml[0][i][c] - ref);
    mul = exp_near(m - ref);
    acc.put(lds[w], mul / sum, c, h);
    m = mx;
    l = sum;
    __syncthreads();
    fa_write<T, D, SPLIT>(Ob, q0, nq, &lds[0][0], 2 * Tile::FLOATS, threadIdx.x, 64 * SPLIT);
  } else {
    wave_fence();
    acc.put(lds[w], 1.0f / l, c, h);
    wave_fence();
    fa_write<T, D, 1>(Ob, q0, nq, lds[w], 0, lane, 64);
  }
  // a row whose every score is -inf has no softmax: NaN, as its outputs
  if (L != nullptr && h == 0 && (SPLIT == 1 || w == 0) && qi < nq)
    L[bh * nq + qi] = m == -INFINITY ? __builtin_nanf("") : m + logf(l);
}

// dq (and D_m = rowsum(o do) to delta_out, if given).
template <typename T, int D, int SPLIT>
__global__ __launch_bounds__(64 * kFaWaves<SPLIT>, D <= 64 ? 2 : 1) void fa_bwd_dq_f32(
    const T *__restrict__ Q, const T *__restrict__ K, const T *__restrict__ V, const T *__restrict__ O,
    const T *__restrict__ dO, const float *__restrict__ L, T *__restrict__ dQ, float *__restrict__ delta_out,
    uint32_t nq, uint32_t nk, float scale, int causal, int kv_group, int nqb) {
  using Tile = FaTile<T, D>;
  __shared__ __attribute__((aligned(16))) float lds[kFaWaves<SPLIT>][2 * Tile::FLOATS];
  // wave-uniform, so that the tile loop and its masks are scalar branches
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  int qb;
  int64_t bh;
  if (!fa_unit<SPLIT>(w, nqb, qb, bh)) return;
  if (causal) qb = nqb - 1 - qb;
  const uint32_t q0 = 32u * qb, qi = q0 + c;
  const T *Kb = K + (bh / kv_group) * nk * D, *Vb = V + (bh / kv_group) * nk * D;
  float *kt = lds[w], *vt = lds[w] + Tile::FLOATS;

  const uint32_t kend = causal ? min(nk, min(q0 + 32, nq)) : nk;
  const int tiles = static_cast<int>((kend + 31) / 32);
  const uint32_t last = causal ? min(kend - 1, qi) : kend - 1;
  int t = SPLIT == 1 ? 0 : w;
  // every first load before anything waits for one
  f32x4 q[D / 8], g[D / 8];
  Tile ts;
  float delta = 0.0f;
  bool odd = false;  // whether the K tile, one with masked pairs, holds an infinity or NaN
  auto diag = [&](int i) { return causal && 32u * i + 31 > q0; };
  auto store_k = [&](int i) {
    if (diag(i)) odd = ts.template store<true>(kt, 32u * i, nk, lane);
    else ts.store(kt, 32u * i, nk, lane);
  };
  const float lse = L[bh * nq + min(qi, nq - 1)];
  {
    f32x4 o[D / 8];
    Tile tv;
    if (t < tiles) {
      tv.fetch(Vb, 32u * t, nk, lane);
      ts.fetch(Kb, 32u * t, nk, lane);
    }
    fa_cols<T, D>(o, O + bh * nq * D, q0, nq, c, h);
    fa_cols<T, D>(g, dO + bh * nq * D, q0, nq, c, h);
    fa_cols<T, D>(q, Q + bh * nq * D, q0, nq, c, h);
    if (t < tiles) {
      tv.store(vt, 32u * t, nk, lane);
      store_k(t);
      wave_fence();
    }
#pragma unroll
    for (int j = 0; j < D / 8; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) delta = __builtin_fmaf(o[j][i], g[j][i], delta);
  }
  delta += other_half(delta);
  if (delta_out != nullptr && h == 0 && (SPLIT == 1 || w == 0) && qi < nq) delta_out[bh * nq + qi] = delta;

  FaAcc<D> dq;
  dq.zero();
  // one set of staging registers: V's next tile is in flight during the first
  // two products, K's during the last
  for (; t < tiles; t += SPLIT) {
    const uint32_t k0 = 32u * t;
    const bool more = t + SPLIT < tiles;
    if (more) ts.fetch(Vb, k0 + 32 * SPLIT, nk, lane);
    f32x16 s = fa_inner<D>(kt, q, c, h);
    const f32x16 dp = fa_inner<D>(vt, g, c, h);
    wave_fence();
    if (more) {
      ts.store(vt, k0 + 32 * SPLIT, nk, lane);
      ts.fetch(Kb, k0 + 32 * SPLIT, nk, lane);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = exp_near(__builtin_fmaf(s[r], scale, -lse)) * (dp[r] - delta);
    if (diag(t) || k0 + 32 > kend) {
      asm volatile("" ::: "memory");  // a branch: whole tiles compare nothing
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = k0 + 8 * (r / 4) + 4 * h + r % 4 > last ? 0.0f : s[r];
    }
    if (diag(t) && __any(odd))
      dq.masked_outer(kt, s, h, [&](int row) { return k0 + row <= last; });
    else
      dq.outer(kt, s, c, h);
    wave_fence();
    if (more) {
      store_k(t + SPLIT);
      wave_fence();
    }
  }
  T *out = dQ + bh * nq * D;
  wave_fence();
  dq.put(lds[w], scale, c, h);
  if constexpr (SPLIT > 1) {
    __syncthreads();
    fa_write<T, D, SPLIT>(out, q0, nq, &lds[0][0], 2 * Tile::FLOATS, threadIdx.x, 64 * SPLIT);
  } else {
    wave_fence();
    fa_write<T, D, 1>(out, q0, nq, lds[w], 0, lane, 64);
  }
}

// dk and dv: columns are keys, tiles the queries of every head that shares
// them.  delta: D_m of every query row, or null (computed here per tile).
template <typename T, int D, int SPLIT>
__global__ __launch_bounds__(64 * kFaWaves<SPLIT>, D <= 64 ? 2 : 1) void fa_bwd_dkv_f32(
    const T *__restrict__ Q, const T *__restrict__ K, const T *__restrict__ V, const T *__restrict__ O,
    const T *__restrict__ dO, const float *__restrict__ L, const float *__restrict__ delta, T *__restrict__ dK,
    T *__restrict__ dV, uint32_t nq, uint32_t nk, float scale, int causal, int kv_group, int nkb) {
  using Tile = FaTile<T, D>;
  __shared__ __attribute__((aligned(16))) float lds[kFaWaves<SPLIT>][2 * Tile::FLOATS];
  __shared__ __attribute__((aligned(16))) float rows[kFaWaves<SPLIT>][2][32];  // lse, D_m of the tile's queries
  // wave-uniform, so that the tile loop and its masks are scalar branches
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  int kb;
  int64_t hkv;
  if (!fa_unit<SPLIT>(w, nkb, kb, hkv)) return;
  const uint32_t c0 = 32u * kb, key = c0 + c;
  float *qt = lds[w], *gt = lds[w] + Tile::FLOATS;

  f32x4 kc[D / 8], vc[D / 8];
  fa_cols<T, D>(kc, K + hkv * nk * D, c0, nk, c, h);
  fa_cols<T, D>(vc, V + hkv * nk * D, c0, nk, c, h);
  FaAcc<D> dk, dv;
  dk.zero();
  dv.zero();
  const int first = causal ? kb : 0, per_head = max(0, static_cast<int>((nq + 31) / 32) - first);
  const int64_t tiles = static_cast<int64_t>(per_head) * kv_group;
  int64_t t = SPLIT == 1 ? 0 : w;
  // one set of staging registers: dO's next tile is in flight during the
  // first three products, Q's during the last
  Tile ts;
  float row_lse = 0.0f, row_delta = 0.0f;
  bool odd_q = false, odd_g = false;  // as in dq, of the dO and Q tiles
  auto head = [&](int64_t i) { return hkv * kv_group + i / per_head; };
  auto query = [&](int64_t i) { return 32u * (first + static_cast<int>(i % per_head)); };
  auto diag = [&](uint32_t q0) { return causal && q0 < c0 + 31; };
  auto fetch_g = [&](int64_t i) {
    const int64_t row = head(i) * nq + min(query(i) + c, nq - 1);
    ts.fetch(dO + head(i) * nq * D, query(i), nq, lane);
    row_lse = L[row];
    if (delta != nullptr) {
      row_delta = delta[row];
    } else {
      const T *o = O + row * D + 4 * h, *g = dO + row * D + 4 * h;
      float s = 0.0f;
      for (int d = 0; d < D; d += 8) {
        const f32x4 a = fa_load4(o + d), b = fa_load4(g + d);
        for (int j = 0; j < 4; ++j) s = __builtin_fmaf(a[j], b[j], s);
      }
      row_delta = s + other_half(s);
    }
  };
  auto store_g = [&](uint32_t q0) {
    if (diag(q0)) odd_g = ts.template store<true>(gt, q0, nq, lane);
    else ts.store(gt, q0, nq, lane);
    if (h == 0) rows[w][0][c] = q0 + c < nq ? row_lse : INFINITY;  // p = 0 past the last query
    else rows[w][1][c] = row_delta;
  };
  auto fetch_q = [&](int64_t i) { ts.fetch(Q + head(i) * nq * D, query(i), nq, lane); };
  auto store_q = [&](uint32_t q0) {
    if (diag(q0)) odd_q = ts.template store<true>(qt, q0, nq, lane);
    else ts.store(qt, q0, nq, lane);
  };
  if (t < tiles) {  // both first tiles in flight together
    fetch_g(t);
    Tile tq;
    tq.fetch(Q + head(t) * nq * D, query(t), nq, lane);
    store_g(query(t));
    ts = tq;
    store_q(query(t));
    wave_fence();
  }
  for (; t < tiles; t += SPLIT) {
    const uint32_t q0 = query(t);
    const bool more = t + SPLIT < tiles, masks = diag(q0), redo_g = masks && __any(odd_g),
               redo_q = masks && __any(odd_q);
    if (more) fetch_g(t + SPLIT);
    f32x16 p = fa_inner<D>(qt, kc, c, h);
    f32x16 ds = fa_inner<D>(gt, vc, c, h);
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const f32x4 lse = *reinterpret_cast<const f32x4 *>(&rows[w][0][8 * r4 + 4 * h]);
      const f32x4 dm = *reinterpret_cast<const f32x4 *>(&rows[w][1][8 * r4 + 4 * h]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 4 * r4 + i;
        p[r] = exp_near(__builtin_fmaf(p[r], scale, -lse[i]));
        ds[r] = p[r] * (ds[r] - dm[i]);
      }
    }
    if (masks || q0 + 32 > nq) {
      asm volatile("" ::: "memory");  // a branch: whole tiles compare nothing
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint32_t qi = q0 + 8 * (r / 4) + 4 * h + r % 4;
        const bool out = (masks && qi < key) || qi >= nq;
        p[r] = out ? 0.0f : p[r];
        ds[r] = out ? 0.0f : ds[r];
      }
    }
    auto seen = [&](int row) { return q0 + row >= key && q0 + row < nq; };
    if (redo_g) dv.masked_outer(gt, p, h, seen);
    else dv.outer(gt, p, c, h);
    wave_fence();
    if (more) {
      store_g(query(t + SPLIT));
      fetch_q(t + SPLIT);
    }
    if (redo_q) dk.masked_outer(qt, ds, h, seen);
    else dk.outer(qt, ds, c, h);
    wave_fence();
    if (more) {
      store_q(query(t + SPLIT));
      wave_fence();
    }
  }
  wave_fence();
  dk.put(lds[w], scale, c, h);
  dv.put(lds[w] + Tile::FLOATS, 1.0f, c, h);
  T *dk_out = dK + hkv * nk * D, *dv_out = dV + hkv * nk * D;
  if constexpr (SPLIT > 1) {
    __syncthreads();
    fa_write<T, D, SPLIT>(dk_out, c0, nk, &lds[0][0], 2 * Tile::FLOATS, threadIdx.x, 64 * SPLIT);
    fa_write<T, D, SPLIT>(dv_out, c0, nk, &lds[0][Tile::FLOATS], 2 * Tile::FLOATS, threadIdx.x, 64 * SPLIT);
  } else {
    wave_fence();
    fa_write<T, D, 1>(dk_out, c0, nk, lds[w], 0, lane, 64);
    fa_write<T, D, 1>(dv_out, c0, nk, lds[w] + Tile::FLOATS, 0, lane, 64);
  }
}

// Waves that share a column block.  Eight for a grid of at most one block per
// CU, which four would leave at one wave per SIMD, if there are tiles for
// them (four / eight waves in us: 16 heads of 500 queries x 2000 keys x 64,
// forward 58.3 / 50.1, dq 70.0 / 64.5; all three kernels of 4 heads of 1000 x
// 1000 x 64 123 / 113, 2 of 1024 x 1024 x 16 60 / 47, but 16 of 200 x 200 x 64
// 41.3 / 42.5).
inline int fa_f32_split(int64_t blocks, int64_t tiles, int D) {
  const int64_t cus = device_cu_count();
  if (blocks <= cus && tiles >= 12 && D <= 64) return 8;
  return blocks < 8 * cus && tiles > 1 ? 4 : 1;
}

// Blocks of 32 columns over `heads`: a workgroup per block, or per four (split 1).
template <typename K, typename... A>
inline void fa_f32_launch(K kernel, int64_t cols, int64_t heads, int split, hipStream_t s, A... args) {
  const unsigned blocks = static_cast<unsigned>(cdiv(cols, 32));
  const dim3 grid(split > 1 ? blocks : (blocks + 3) / 4, static_cast<unsigned>(heads));
  hipLaunchKernelGGL(kernel, grid, dim3(64 * (split == 1 ? 4 : split)), 0, s, args..., static_cast<int>(blocks));
}

// Where the per-row kernels (a wave per query or key row, its lanes the rows of
// the other side) are the faster ones, though a wave here does the same for 32
// columns: with most of the 32 missing, on a chip that the blocks fill, and with
// so little of everything that the way to the first product counts.  Measured in
// us, rows / here, forward, fp32 (heads x queries x keys x head_dim): 2048 x 1 x
// 1024 x 16 83 / 129, x 128 427 / 1573, 4096 x 2 x 512 x 64 367 / 441, 1024 x 1 x
// 64 x 64 7.2 / 16, but 1024 x 1 x 512 x 64 60 / 55 (the tiles shared by four
// waves), 2048 x 4 x 256 x 64 175 / 112; 8 x 16 x 64 x 128 7.1 / 10.2, 32 x 16 x
// 64 x 32 4.2 / 4.5, 32 x 33 x 32 x 128 8.5 / 10.7 (the call's host time in it),
// but 128 x 8 x 64 x 128 14.9 / 10.1.  dq gains up to twice the keys, 1536 x 1 x
// 512 x 16 25 / 38, but not for two queries at head_dim 32 and 64, 2048 x 2 x 512
// x 64 314 / 278.  dk/dv 8 x 8 x 64 x 64 8.6 / 10.7, 1024 x 1 x 1 x 64 8.7 / 18.5,
// but 128 x 16 x 16 x 64 27.8 / 9.7.
//
// Forward and dq: BH heads of nq queries, which see at most nk keys.
inline bool fa_rows_q(bool dq, bool f32, int64_t BH, int64_t nq, int64_t nk, int D) {
  const int64_t cus = device_cu_count();
  if (nk <= 64 && BH * nq * std::max<int64_t>(nk, 16) <= (!dq && D == 128 && nk <= 32 ? 65536 : 32768)) return true;
  if (BH < 2 * cus) return false;
  if (BH >= 8 * cus) {
    const bool four = f32 ? !dq && D == 128 : D == 16, one = f32 && dq && (D == 32 || D == 64);
    if (nq <= (four ? 4 : one ? 1 : 2)) return true;
  }
  if (nq > 4) return nq * std::max<int64_t>(nk, 8) <= D;
  if (nq > 1) return nk <= (nq > 2 ? std::max<int64_t>(16, D / nq) : 64);
  return nk <= (dq && D <= 32 && BH >= 3 * cus ? 512 : dq || BH >= 4 * cus ? 256 : 128);
}

// dk/dv: K/V heads of nk keys, nq queries of all heads that share them.
inline bool fa_rows_k(bool f32, int64_t heads, int64_t nq, int64_t nk, int D) {
  if ((f32 || D != 32) && (nq <= 8 ? heads * nk <= 1024 : nq <= 16 && heads * nk <= 256)) return true;
  return heads >= 2 * device_cu_count() && nk * std::max<int64_t>(nq, 8) <= 16;
}

// The kernel template NAME<T, D, SPLIT> for a split (8: D <= 64 only).
#define TEENY_FA_F32(NAME, T, D, split) \
  ((split) == 8 ? NAME<T, D, (D <= 64 ? 8 : 4)> : (split) == 4 ? NAME<T, D, 4> : NAME<T, D, 1>)

}  // namespace teeny
