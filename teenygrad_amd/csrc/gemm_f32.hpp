// fp32 GEMM on the fp32 matrix cores: linear_forward / linear_backward in fp32.
//
//   C[m,n] = sum_k A[m,k] B[n,k] (+ bias[n]), every operand with two strides,
// one of A's and one of B's being 1 (the forward reads both along k, dx reads
// w along its other axis, dw both).  v_mfma_f32_32x32x2_f32: fp32 products
// and sums, as the FMA loop it takes the place of.
//
// Bound: the fp32 matrix cores (157 TFLOP/s, 64 cycles per 4096 FLOP and
// SIMD), or for few rows the weights' bytes.  One 32 x 32 MFMA wants only
// 512 bytes of LDS reads per 64 cycles, so small wave tiles are no loss, and
// the tile is picked to fill the chip: 64 x 64 with eight waves (2 x 2
// quadrants, two waves per quadrant on alternate k's, so that each SIMD has
// two waves even at one workgroup per CU), 128 x 128 once those fill it too
// (half the L2 bytes), 32 x 64 for up to 32 rows.  Grids that leave CUs idle
// split K into fp32 slices in the stream's workspace, added in slice order.
// Operands go global -> registers (two chunks of 32 k ahead) -> LDS (double
// buffered, one barrier per chunk).  An operand contiguous along k sits in
// LDS as [row][36] and a fragment is one 16-byte read of four k's; one
// contiguous along its rows sits as [k][rows + 8] and is read as four words:
// both layouts are free of bank conflicts and neither needs a transpose.
// 4-byte alignment is enough (global dwordx4 loads); the ragged last vector
// of a row is read shifted back into the row and shifted in registers.
// Measured (forward + dx + dw + db of one layer, M x N x K): 1000 x 1024 x
// 1024 522 us with the FMA tile kernel -> 81 us (78 TFLOP/s with db and the
// four launches; a 64 x 64 tile per CU, K = 1024, cannot take less than 14
// us), 2048^3 493 us (105 TFLOP/s), 4096^3 3170 us (130 TFLOP/s).
#pragma once

#include "mfma.hpp"

namespace teeny {

struct GemmF32Params {
  const float *A, *B;
  float *C;            // output, or the partial slices [splits][M][N]
  const float *bias;   // [N] or null (null with splits > 1: the reduce adds it)
  int64_t sa, sb;      // stride of the non-contiguous axis
  int64_t scm, scn;    // strides of C
  int64_t slice;       // elements between partial slices
  int M, N, K;
  uint32_t k_len;      // k's per split (a multiple of the chunk: K rounded up, 2^31 at most)
  int tiles_n;
};

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kF32KC = 32;  // k's per chunk

// Rows x 32 k of one operand: global -> registers -> LDS, and the fragments.
template <int ROWS, bool KCONTIG, int NT> struct F32Operand {
  static constexpr int VEC = ROWS * kF32KC / 4;          // 16-byte vectors per chunk
  static constexpr int NV = (VEC + NT - 1) / NT;         // per thread
  static constexpr int LD = KCONTIG ? kF32KC + 4 : ROWS + 8;
  static constexpr int FLOATS = KCONTIG ? ROWS * LD : kF32KC * LD;
  const float *base;
  int64_t s;
  int K, last_row, row0;
  __device__ __forceinline__ void init(const float *p, int64_t stride, int rows, int K_, int row0_) {
    base = p;
    s = stride;
    K = K_;
    last_row = rows - 1;
    row0 = row0_;
  }
  // One vector of the chunk at k0.  TAIL: the chunk may run past K (those
  // k's read as zero in both operands).  Rows past the last only reach
  // outputs that are not stored; they read valid rows.
  template <bool TAIL> __device__ __forceinline__ f32x4 load(int t, int k0) const {
    if constexpr (KCONTIG) {
      const int row = min(row0 + t / (kF32KC / 4), last_row), k = k0 + 4 * (t % (kF32KC / 4));
      const float *p = base + row * s;
      if constexpr (!TAIL) return *reinterpret_cast<const f32x4u *>(p + k);
      const int kk = min(k, K - 4), d = k - kk;
      const f32x4 u = *reinterpret_cast<const f32x4u *>(p + kk);
      return f32x4{d < 1 ? u[0] : d < 2 ? u[1] : d < 3 ? u[2] : d < 4 ? u[3] : 0.0f,
                   d < 1 ? u[1] : d < 2 ? u[2] : d < 3 ? u[3] : 0.0f,
                   d < 1 ? u[2] : d < 2 ? u[3] : 0.0f, d < 1 ? u[3] : 0.0f};
    } else {
      const int r = row0 + 4 * (t % (ROWS / 4)), k = k0 + t / (ROWS / 4);
      const int rr = min(r, last_row - 3), d = r - rr;
      const float *p = base + (TAIL ? min(k, K - 1) : k) * s + rr;
      f32x4 u = *reinterpret_cast<const f32x4u *>(p);
      u = f32x4{d < 1 ? u[0] : d < 2 ? u[1] : d < 3 ? u[2] : u[3], d < 1 ? u[1] : d < 2 ? u[2] : u[3],
                d < 1 ? u[2] : u[3], u[3]};
      if constexpr (TAIL) {
        if (k >= K) u = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      }
      return u;
    }
  }
  template <bool TAIL> __device__ __forceinline__ void fetch(f32x4 (&r)[NV], int tid, int k0) const {
#pragma unroll
    for (int i = 0; i < NV; ++i)
      if (VEC % NT == 0 || tid + i * NT < VEC) r[i] = load<TAIL>(tid + i * NT, k0);
  }
  __device__ __forceinline__ static void store(float *lds, const f32x4 (&r)[NV], int tid) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int t = tid + i * NT;
      if (VEC % NT == 0 || t < VEC) {
        if constexpr (KCONTIG)
          *reinterpret_cast<f32x4 *>(lds + t / (kF32KC / 4) * LD + 4 * (t % (kF32KC / 4))) = r[i];
        else
          *reinterpret_cast<f32x4 *>(lds + t / (ROWS / 4) * LD + 4 * (t % (ROWS / 4))) = r[i];
      }
    }
  }
  // k's kb .. kb + 3 of `row`
  __device__ __forceinline__ static f32x4 frag(const float *lds, int row, int kb) {
    if constexpr (KCONTIG) return *reinterpret_cast<const f32x4 *>(lds + row * LD + kb);
    else return f32x4{lds[kb * LD + row], lds[(kb + 1) * LD + row], lds[(kb + 2) * LD + row], lds[(kb + 3) * LD + row]};
  }
};

template <int BM, int BN, int WM, int WN, int WK, bool AK, bool BKC>
__global__ __launch_bounds__(64 * WM * WN * WK) void gemm_f32_mfma(GemmF32Params p) {
  constexpr int NT = 64 * WM * WN * WK;
  constexpr int MI = BM / WM / 32, NI = BN / WN / 32;
  using OA = F32Operand<BM, AK, NT>;
  using OB = F32Operand<BN, BKC, NT>;
  constexpr int STAGE = OA::FLOATS + OB::FLOATS;
  constexpr int RED = (WK - 1) * WM * WN * MI * NI * 1024;  // the k-split waves' sums
  __shared__ __attribute__((aligned(16))) float lds[2 * STAGE > RED ? 2 * STAGE : RED];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, h = lane >> 5, c = lane & 31;
  const int wk = w % WK, wn = w / WK % WN, wm = w / WK / WN;
  const int tile = xcd_remap(blockIdx.x, gridDim.x);
  const int m0 = tile / p.tiles_n * BM, n0 = tile % p.tiles_n * BN;
  // K may be 2^31 - 1: no end past K is formed, and rounded-up counts are unsigned
  const int kb = static_cast<int>(blockIdx.y * p.k_len);
  const uint32_t k_count = min(static_cast<uint32_t>(p.K - kb), p.k_len);
  OA a;
  OB b;
  a.init(p.A, p.sa, p.M, p.K, m0);
  b.init(p.B, p.sb, p.N, p.K, n0);

  f32x16 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = zero16();

  const int n_chunks = static_cast<int>((k_count + kF32KC - 1) / kF32KC);
  f32x4 ra[2][OA::NV], rb[2][OB::NV];
  auto fetch = [&](int set, int chunk) {
    if (chunk >= n_chunks) return;
    const int k0 = kb + chunk * kF32KC;
    if (static_cast<uint32_t>(k0) + kF32KC <= static_cast<uint32_t>(p.K)) {
      a.template fetch<false>(ra[set], tid, k0);
      b.template fetch<false>(rb[set], tid, k0);
    } else {
      a.template fetch<true>(ra[set], tid, k0);
      b.template fetch<true>(rb[set], tid, k0);
    }
  };
  auto stash = [&](int set) {
    OA::store(lds + set * STAGE, ra[set], tid);
    OB::store(lds + set * STAGE + OA::FLOATS, rb[set], tid);
  };
  fetch(0, 0);
  fetch(1, 1);
  stash(0);
  fetch(0, 2);
  __syncthreads();
  // FULL: the next chunk and the one three ahead exist and are whole, so
  // their code has no branch (behind one the compiler waits for every load)
  auto step = [&](auto set_, auto full_, int chunk) {
    constexpr int set = decltype(set_)::value;
    if constexpr (decltype(full_)::value) {
      stash(set ^ 1);
      a.template fetch<false>(ra[set ^ 1], tid, kb + (chunk + 3) * kF32KC);
      b.template fetch<false>(rb[set ^ 1], tid, kb + (chunk + 3) * kF32KC);
    } else {
      if (chunk + 1 < n_chunks) stash(set ^ 1);
      fetch(set ^ 1, chunk + 3);
    }
    const float *la = lds + set * STAGE, *lb = la + OA::FLOATS;
#pragma unroll
    for (int j = 0; j < kF32KC / 8 / WK; ++j) {
      const int k8 = 8 * (j * WK + wk) + 4 * h;
      f32x4 fa[MI], fb[NI];
#pragma unroll
      for (int i = 0; i < MI; ++i) fa[i] = OA::frag(la, (wm * MI + i) * 32 + c, k8);
#pragma unroll
      for (int i = 0; i < NI; ++i) fb[i] = OB::frag(lb, (wn * NI + i) * 32 + c, k8);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int l = 0; l < NI; ++l)
            acc[i][l] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][s], fb[l][s], acc[i][l], 0, 0, 0);
    }
    __syncthreads();
  };
  constexpr std::integral_constant<int, 0> s0{};
  constexpr std::integral_constant<int, 1> s1{};
  const int n_full = static_cast<int>(k_count / kF32KC);
  int ch = 0;
  for (; ch + 4 < n_full; ch += 2) {
    step(s0, std::true_type{}, ch);
    step(s1, std::true_type{}, ch + 1);
  }
  for (; ch + 1 < n_chunks; ch += 2) {
    step(s0, std::false_type{}, ch);
    step(s1, std::false_type{}, ch + 1);
  }
  if (ch < n_chunks) step(s0, std::false_type{}, ch);

  // sums of the waves that share a quadrant meet in LDS (the last step ended with a barrier)
  if constexpr (WK > 1) {
    if (wk > 0) {
      float *red = lds + ((wk - 1) * WM * WN + wm * WN + wn) * MI * NI * 1024;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int l = 0; l < NI; ++l)
#pragma unroll
          for (int r = 0; r < 16; ++r) red[((i * NI + l) * 16 + r) * 64 + lane] = acc[i][l][r];
    }
    __syncthreads();
    if (wk > 0) return;
#pragma unroll
    for (int q = 1; q < WK; ++q) {
      const float *red = lds + ((q - 1) * WM * WN + wm * WN + wn) * MI * NI * 1024;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int l = 0; l < NI; ++l)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][l][r] += red[((i * NI + l) * 16 + r) * 64 + lane];
    }
  }
  float *C = p.C + blockIdx.y * p.slice;
#pragma unroll
  for (int l = 0; l < NI; ++l) {
    const int n = n0 + (wn * NI + l) * 32 + c;
    if (n >= p.N) continue;
    const float bias = p.bias != nullptr ? p.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + (wm * MI + i) * 32 + 8 * (r / 4) + 4 * h + r % 4;
        if (m < p.M) C[m * p.scm + n * p.scn] = p.bias != nullptr ? acc[i][l][r] + bias : acc[i][l][r];
      }
  }
}

// C = the slices' sum in slice order (+ bias).
__global__ __launch_bounds__(256) void gemm_f32_splitk_sum(const float *__restrict__ part, int splits, int64_t slice,
                                                           float *__restrict__ C, int64_t scm, int64_t scn,
                                                           const float *__restrict__ bias, int64_t total, int N) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= total) return;
  float v = part[i];
  int s = 1;
  for (; s + 3 < splits; s += 4) {
    const float a = part[i + s * slice], b = part[i + (s + 1) * slice], c = part[i + (s + 2) * slice],
                d = part[i + (s + 3) * slice];
    v = v + a;
    v = v + b;
    v = v + c;
    v = v + d;
  }
  for (; s < splits; ++s) v += part[i + s * slice];
  const int64_t m = i / N, n = i - m * N;
  C[m * scm + n * scn] = bias != nullptr ? v + bias[n] : v;
}

struct GemmF32Plan {
  int bm, bn, splits;
  uint32_t k_len;
};

// Tile and split for one GEMM.  scratch: bytes of workspace that may hold slices.
inline GemmF32Plan gemm_f32_plan(int64_t M, int64_t N, int64_t K, size_t scratch) {
  const int cus = device_cu_count();
  GemmF32Plan pl{64, 64, 1, static_cast<uint32_t>(cdiv(K, kF32KC) * kF32KC)};
  if (M <= 32) pl.bm = 32;
  else if (cdiv(M, 128) * cdiv(N, 128) >= 2 * cus) pl.bm = pl.bn = 128;
  const int64_t tiles = cdiv(M, pl.bm) * cdiv(N, pl.bn);
  // idle CUs: split K, at least four chunks to a split, to about two workgroups per CU
  if (tiles < cus) {
    int64_t s = std::min<int64_t>(cdiv(2 * cus, tiles), K / (4 * kF32KC));
    s = std::min<int64_t>(s, static_cast<int64_t>(scratch / (static_cast<size_t>(M) * N * 4)));
    if (s > 1) {
      const int64_t chunks = cdiv(cdiv(K, kF32KC), s);
      pl.k_len = static_cast<uint32_t>(chunks * kF32KC);
      pl.splits = static_cast<int>(cdiv(K, pl.k_len));
    }
  }
  return pl;
}

// Workspace bytes of the plan that has all it wants.
inline size_t gemm_f32_scratch_bytes(int64_t M, int64_t N, int64_t K) {
  const GemmF32Plan pl = gemm_f32_plan(M, N, K, ~size_t{0});
  return pl.splits > 1 ? static_cast<size_t>(pl.splits) * M * N * 4 : 0;
}

// Whether the kernel reads these operands: one unit stride each, and four of
// whatever a 16-byte load spans.
inline bool gemm_f32_ok(int64_t sam, int64_t sak, int64_t sbn, int64_t sbk, int64_t M, int64_t N, int64_t K) {
  const bool ok_a = sak == 1 ? K >= 4 : (sam == 1 && M >= 4);
  const bool ok_b = sbk == 1 ? K >= 4 : (sbn == 1 && N >= 4);
  // rows beyond the generic kernel's grid are its to refuse; 2^32 threads in a grid
  return ok_a && ok_b && K >= 1 && cdiv(M, 64) <= 65535 && cdiv(M, 32) * cdiv(N, 64) < (int64_t{1} << 32) / 512;
}

template <bool AK, bool BKC> inline void gemm_f32_launch(const GemmF32Plan &pl, const GemmF32Params &p, hipStream_t s) {
  const dim3 grid(static_cast<unsigned>(cdiv(p.M, pl.bm) * cdiv(p.N, pl.bn)), static_cast<unsigned>(pl.splits));
  if (pl.bm == 32) hipLaunchKernelGGL((gemm_f32_mfma<32, 64, 1, 2, 4, AK, BKC>), grid, dim3(512), 0, s, p);
  else if (pl.bm == 64) hipLaunchKernelGGL((gemm_f32_mfma<64, 64, 2, 2, 2, AK, BKC>), grid, dim3(512), 0, s, p);
  else hipLaunchKernelGGL((gemm_f32_mfma<128, 128, 2, 4, 1, AK, BKC>), grid, dim3(512), 0, s, p);
}

inline void launch_gemm_f32(const float *A, int64_t sam, int64_t sak, const float *B, int64_t sbn, int64_t sbk,
                            float *C, int64_t scm, int64_t scn, const float *bias, int64_t M, int64_t N, int64_t K,
                            hipStream_t s, const Scratch &scratch) {
  const GemmF32Plan pl = gemm_f32_plan(M, N, K, scratch.ptr != nullptr ? scratch.bytes : 0);
  const bool ak = sak == 1, bk = sbk == 1, split = pl.splits > 1;
  GemmF32Params p{};
  p.A = A;
  p.B = B;
  p.C = split ? static_cast<float *>(scratch.ptr) : C;
  p.bias = split ? nullptr : bias;
  p.sa = ak ? sam : sak;
  p.sb = bk ? sbn : sbk;
  p.scm = split ? N : scm;
  p.scn = split ? 1 : scn;
  p.slice = split ? M * N : 0;
  p.M = static_cast<int>(M);
  p.N = static_cast<int>(N);
  p.K = static_cast<int>(K);
  p.k_len = pl.k_len;
  p.tiles_n = static_cast<int>(cdiv(N, pl.bn));
  if (ak && bk) gemm_f32_launch<true, true>(pl, p, s);
  else if (ak) gemm_f32_launch<true, false>(pl, p, s);
  else if (bk) gemm_f32_launch<false, true>(pl, p, s);
  else gemm_f32_launch<false, false>(pl, p, s);
  if (split)
    hipLaunchKernelGGL(gemm_f32_splitk_sum, dim3(static_cast<unsigned>(cdiv(M * N, 256))), dim3(256), 0, s, p.C,
                       pl.splits, p.slice, C, scm, scn, bias, M * N, p.N);
}

}  // namespace teeny
