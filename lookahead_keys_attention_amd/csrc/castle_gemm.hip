// Products of a layer's projections over some hundreds to some thousands of rows:
//   forward          y[R, N]  = x[R, K] w[N, K]^T          both operands contraction-contiguous
//   input gradient   dx[R, K] = dy[R, N] w[N, K]           the second one stored [contraction][free]
//   weight gradient  dw[N, K] = dy[R, N]^T x[R, K]         both stored [contraction][free]
//
// Why own kernels: a call of the library's product costs 18 us of host time, more than the whole product takes on the GPU
// up to about 5 GFLOP, and its weight gradient walks all rows in one chain per output tile (1536 x 256 from 3000
// rows: 30 us).  A launch here costs 4 us of host time, the rows of a weight gradient are split over workgroups, and GELU
// and its derivative ride on the store.
//
// Four waves share a BM x BN tile of the output (2 x 2 quarters).  What bounds these sizes is latency: few workgroups on
// a CU and a short contraction.  So the pieces of two steps of the contraction are in flight in registers while a third
// is in LDS (two buffers, one barrier a step).  Operands stored [contraction][free] are copied as they are and
// read with transpose reads.
#include "castle_tiles.h"
#include "castle_dispatch.h"
#include "castle_gemm.h"
#include <algorithm>
#include "castle_rows.h"

namespace castle {
namespace {

// Phi(x) = erfc(-x / sqrt 2) / 2.  For 16-bit outputs from the Chebyshev fit of Numerical Recipes (erfcc, fractional error
// below 1.2e-7 everywhere); the library's erff takes three times the instructions, which a store of 16384 x 2048 felt
// with 8 us.
template <typename T> __device__ __forceinline__ float normal_cdf(float x) {
  if constexpr (sizeof(T) == 4) {
    return 0.5f * (1.f + erff(x * 0.70710678f));
  } else {
    const float z = fabsf(x) * 0.70710678f, t = fast_rcp(__builtin_fmaf(0.5f, z, 1.f));
    float p = 0.17087277f;
    p = __builtin_fmaf(p, t, -0.82215223f);
    p = __builtin_fmaf(p, t, 1.48851587f);
    p = __builtin_fmaf(p, t, -1.13520398f);
    p = __builtin_fmaf(p, t, 0.27886807f);
    p = __builtin_fmaf(p, t, -0.18628806f);
    p = __builtin_fmaf(p, t, 0.09678418f);
    p = __builtin_fmaf(p, t, 0.37409196f);
    p = __builtin_fmaf(p, t, 1.00002368f);
    p = __builtin_fmaf(p, t, -1.26551223f);
    const float e = 0.5f * t * fast_exp2(kLog2e * (p - z * z));
    return x < 0.f ? e : 1.f - e;
  }
}
template <typename T> __device__ __forceinline__ float gelu(float x) { return x * normal_cdf<T>(x); }
template <typename T> __device__ __forceinline__ float gelu_slope(float x) {
  return normal_cdf<T>(x) + x * 0.3989422804f * fast_exp2(-0.5f * kLog2e * x * x);
}

// A tile of FREE rows / columns and BK steps of the contraction: global -> registers -> LDS -> operand fragments.
// KC: the operand is contraction-contiguous (LDS [FREE][BK]), else stored [contraction][free] (LDS [BK][FREE]).
template <typename T, bool KC, int FREE, int BK, int G> struct Operand {
  static constexpr int V = elem_traits<T>::vec16;
  static constexpr int COLS = KC ? BK : FREE, ROWS = KC ? FREE : BK, VPR = COLS / V, N = ROWS * VPR / kThreads;
  static constexpr int LD = KC ? lds_ld<T>(COLS) : lds_ld_tr<T>(COLS), ELEMS = ROWS * LD;
  static_assert(ROWS * VPR % kThreads == 0, "a whole number of pieces per thread");
  typedef vec<T, V> vt;
  // where the pieces of this thread are, in elements from the operand's start: one addition per piece and step (formed
  // from row and column each time they took longer than the products).  Pieces beyond the free end read another row's
  // data: those outputs are not stored.
  int at[N];
  vt r[2][N];
  static __device__ __forceinline__ int row_of(int j) { return (threadIdx.x % kThreads + j * kThreads) / VPR; }
  static __device__ __forceinline__ int col_of(int j) { return (threadIdx.x % kThreads + j * kThreads) % VPR * V; }
  __device__ __forceinline__ void start(int ld, int free0, int free_end, int k0) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int f = free0 + (KC ? row_of(j) : col_of(j)), k = k0 + (KC ? col_of(j) : row_of(j));
      at[j] = KC ? min(f, free_end - 1) * ld + k : k * ld + (f < free_end ? f : 0);
    }
  }
  __device__ __forceinline__ void load(int slot, const T* p, int ld, int k, int k_end) {
    if (k + BK <= k_end) {
#pragma unroll
      for (int j = 0; j < N; ++j) r[slot][j] = *reinterpret_cast<const vt*>(p + at[j]);
    } else {   // the last step: zeros behind the contraction's end
#pragma unroll
      for (int j = 0; j < N; ++j) {
#pragma unroll
        for (int e = 0; e < V; ++e) r[slot][j][e] = (T)0.f;
        if (k + (KC ? col_of(j) : row_of(j)) < k_end) r[slot][j] = *reinterpret_cast<const vt*>(p + at[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < N; ++j) at[j] += KC ? G * BK : G * BK * ld;
  }
  __device__ __forceinline__ void store(int slot, T* lds) const {
#pragma unroll
    for (int j = 0; j < N; ++j) *reinterpret_cast<vt*>(lds + row_of(j) * LD + col_of(j)) = r[slot][j];
  }
  static __device__ __forceinline__ frag<T> read(const T* lds, int free0, int k0, int c, int g) {
    if constexpr (KC) return ld_nat<T>(lds, LD, free0 + c, k0 + 8 * g);
    else return ld_free<T, false>(lds, LD, free0, FREE, k0, c, g);
  }
};

// G: groups of four waves.  Two take alternate steps of the contraction for the same tile, each in LDS of its own, and are summed at
// the end: where the tiles leave a CU one workgroup, a second wave per SIMD works while the first waits for LDS and barrier.
template <typename T, bool AK, bool BKC, int BM, int BN, int BK, int G>
__global__ __launch_bounds__(kThreads * G, BM == 128 ? 2 : 4) void gemm_kernel(GemmArgs a) {
  constexpr int WM = BM / 64, WN = BN / 64;   // 32-wide pieces of a wave's quarter
  typedef Operand<T, AK, BM, BK, G> OpA;
  typedef Operand<T, BKC, BN, BK, G> OpB;
  constexpr int V = elem_traits<T>::vec16, LDC = BN + V;
  constexpr int kStage = 2 * (OpA::ELEMS + OpB::ELEMS), kOut = BM * LDC;
  __shared__ __attribute__((aligned(16))) T smem[G * kStage > kOut ? G * kStage : kOut];
  const int lane = lane_id(), wave = wave_id() % 4, group = wave_id() / 4, c = lane & 31, g = lane >> 5;
  // Workgroups go round the 8 XCDs, each with an L2 of its own: XCD x takes the x-th eighth of the tiles, so the rows of
  // `a` are read by one XCD, not by all (input gradient of 3000 rows x 1536 x 256: 13.5 -> 11.1 us).  A workgroup takes
  // several tiles where there are more than the CUs hold: the first steps of the next are requested before the
  // output of the last is written.
  const int tiles_n = (a.N + BN - 1) / BN, tiles = (a.M + BM - 1) / BM * tiles_n;
  const int share = (tiles + 7) / 8, first = blockIdx.x % 8 * share, last = min(tiles, first + share);
  const int wm = wave / 2 * (BM / 2), wn = wave % 2 * (BN / 2);
  const int k0 = blockIdx.y * a.k_per_split, k_end = min(a.K, k0 + a.k_per_split);
  const int steps = ((k_end - k0 + BK - 1) / BK + G - 1) / G;   // of a group: its steps are G BK apart
  T* const stage = smem + group * kStage;
  const T *pa = static_cast<const T*>(a.a), *pb = static_cast<const T*>(a.b);
  OpA ra;
  OpB rb;
  acc_t acc[WM][WN];   // [n rows, m lanes]
  int tile = first + blockIdx.x / 8;
  auto request = [&]() __attribute__((always_inline)) {
    ra.start((int)a.lda, tile / tiles_n * BM, a.M, k0 + group * BK);
    rb.start((int)a.ldb, tile % tiles_n * BN, a.N, k0 + group * BK);
#pragma unroll
    for (int p = 0; p < 2; ++p) {   // (a step beyond the end loads zeros)
      ra.load(p, pa, (int)a.lda, k0 + (p * G + group) * BK, k_end);
      rb.load(p, pb, (int)a.ldb, k0 + (p * G + group) * BK, k_end);
    }
  };
  auto step = [&](auto parity, int it) __attribute__((always_inline)) {
    constexpr int p = decltype(parity)::value;
    T* la = stage + p * (OpA::ELEMS + OpB::ELEMS);
    T* lb = la + OpA::ELEMS;
    ra.store(p, la);
    rb.store(p, lb);
    if (it + 2 < steps) {
      ra.load(p, pa, (int)a.lda, k0 + ((it + 2) * G + group) * BK, k_end);
      rb.load(p, pb, (int)a.ldb, k0 + ((it + 2) * G + group) * BK, k_end);
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < BK / 16; ++s) {
      frag<T> fa[WM], fb[WN];
#pragma unroll
      for (int i = 0; i < WM; ++i) fa[i] = OpA::read(la, wm + 32 * i, 16 * s, c, g);
#pragma unroll
      for (int j = 0; j < WN; ++j) fb[j] = OpB::read(lb, wn + 32 * j, 16 * s, c, g);
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) mma(acc[i][j], fb[j], fa[i]);
    }
  };
  const int amax_tile = a.amax_from / BN, amax_tiles = (a.amax_to - 1) / BN + 1 - amax_tile;   // of a row of tiles
  if (a.amax != nullptr && blockIdx.x == 0) {
    for (int i = (a.M + BM - 1) / BM * amax_tiles + threadIdx.x; i < kAmaxBlocks; i += kThreads * G) a.amax[i] = 0.f;
    if (threadIdx.x == 0 && a.amax_status != nullptr) *a.amax_status = 0;
  }
  if (tile < last) request();
  while (tile < last) {
    const int m0 = tile / tiles_n * BM, n0 = tile % tiles_n * BN;
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) zero(acc[i][j]);
    for (int it = 0; it < steps; it += 2) {
      step(std::integral_constant<int, 0>(), it);
      if (it + 1 < steps) step(std::integral_constant<int, 1>(), it + 1);
    }
    if constexpr (G == 2) {
      typedef vec<float, 4> v4;
      static_assert(kThreads * WM * WN * 64 <= (int)sizeof(smem), "one group's sums");
      v4* sums = reinterpret_cast<v4*>(smem);
      asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");   // the loop may end right behind a product
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();   // the operands of the last step are dead
      if (group == 1) {
#pragma unroll
        for (int i = 0; i < WM * WN; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) sums[(i * 4 + q) * kThreads + threadIdx.x % kThreads] = pack4<float>(acc[i / WN][i % WN], q);
      }
      __syncthreads();
      if (group == 0) {
#pragma unroll
        for (int i = 0; i < WM * WN; ++i)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const v4 other = sums[(i * 4 + q) * kThreads + threadIdx.x];
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i / WN][i % WN][4 * q + e] += other[e];
          }
      }
    }
    tile += gridDim.x / 8;
    if (tile < last) request();
    if (a.part != nullptr) {   // partial product of this range of the contraction
      float* part = a.part + (int64_t)blockIdx.y * a.M * a.N;
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int m = m0 + wm + 32 * i + c, n = n0 + wn + 32 * j + 8 * q + 4 * g;
            if (group == 0 && m < a.M && n < a.N) *reinterpret_cast<vec<float, 4>*>(part + (int64_t)m * a.N + n) = pack4<float>(acc[i][j], q);
          }
      __syncthreads();   // the operands of the last step are dead
      continue;
    }
    // through LDS to whole rows
    __syncthreads();
    if (group == 0)
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) st4<T>(smem + (wm + 32 * i + c) * LDC + wn + 32 * j + 8 * q + 4 * g, pack4<T>(acc[i][j], q));
    __syncthreads();
    typedef vec<T, V> vt;
    typedef vec<float, V> vf;
    float most = 0.f;
    for (int i = threadIdx.x; i < BM * (BN / V); i += kThreads * G) {
      const int row = i / (BN / V), col = i % (BN / V) * V, m = m0 + row, n = n0 + col;
      if (m >= a.M || n >= a.N) continue;
      vt x = *reinterpret_cast<const vt*>(smem + row * LDC + col);
      const int64_t at = (int64_t)m * a.ldc + n;
      if (a.epilogue == kGemmGeluSlope) {
        vf f = __builtin_convertvector(x, vf);
        const vf u = __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.aux) + at), vf);
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] *= gelu_slope<T>(u[e]);
        x = __builtin_convertvector(f, vt);
      }
      *reinterpret_cast<vt*>(static_cast<T*>(a.c) + at) = x;
      if (a.amax != nullptr && n >= a.amax_from && n < a.amax_to) {
        const vf f = __builtin_convertvector(x, vf);
#pragma unroll
        for (int e = 0; e < V; ++e) most = fmaxf(most, fabsf(f[e]));   // fmaxf drops NaNs
      }
      if (a.epilogue == kGemmGelu) {
        vf f = __builtin_convertvector(x, vf);
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = gelu<T>(f[e]);
        *reinterpret_cast<vt*>(static_cast<T*>(a.aux) + at) = __builtin_convertvector(f, vt);
      }
    }
    const int slot = n0 / BN - amax_tile;
    if (a.amax != nullptr && slot >= 0 && slot < amax_tiles) {
      __shared__ float s_most[G * kThreads / 64];
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) most = fmaxf(most, __shfl_xor(most, o));
      if (lane == 0) s_most[wave_id()] = most;
      __syncthreads();
      if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < G * kThreads / 64; ++w) most = fmaxf(most, s_most[w]);
        a.amax[m0 / BM * amax_tiles + slot] = fminf(most, 3.0e38f);   // an infinite value counts as the largest finite one
      }
    }
    __syncthreads();
  }
}

// Tile, number of ranges of the contraction and groups of a workgroup, from what a launch takes (us, measured over 96 ... 5916 rows,
// outputs of 128 ... 3072 columns and contractions of 128 ... 5916): 2.3, and per step of a workgroup 0.42 (64 x 64) or 0.95
// (128 x 128) when it has a CU to itself, 0.32 or 0.9 when the CU has others; fp32 0.78 and 0.62.  A second group takes a step of a
// workgroup that has a CU to itself to 0.30, fp32 0.66, for 0.3 at the end (one range, one group / two: 3000 rows of 1536 -> 256
// 12.7 / 9.9, 256 rows of fp32 512 -> 3072 15.1 / 13.1; level at two workgroups a CU, behind from three on: 3000 rows of 256 -> 1536 8.7
// / 11.3).  A split adds a second launch, 2.5, and its partial results, written and read.  Weight gradient of 3000 rows, 1536 x
// 256 out: 22.6 us in one range, 14.1 in two of two groups; 3000 rows 256 -> 1536 forward: 8.4 on 64 x 64 tiles, 9.5 on 128 x 128;
// 5916 rows of 512 -> 2048: 30.6 and 23.2.
struct Plan {
  int tile, splits, groups;
};
Plan plan(int M, int N, int K, bool can_split, int elem_size) {
  Plan best = {64, 1, 1};
  double best_cost = 1e30;
  for (int tile = 64; tile <= (elem_size == 2 ? 128 : 64); tile += 64) {
    const double alone = elem_size == 4 ? 0.78 : tile == 64 ? 0.42 : 0.95, shared = elem_size == 4 ? 0.62 : tile == 64 ? 0.32 : 0.9;
    const int64_t tiles = (int64_t)((M + tile - 1) / tile) * ((N + tile - 1) / tile);
    const int steps = (K * elem_size + 127) / 128;   // 128 bytes of the contraction a step
    for (int s = 1; s <= (can_split ? std::min(16, (steps + 1) / 2) : 1); ++s) {
      const int64_t per_cu = (tiles * s + 255) / 256, n = (steps + s - 1) / s;
      const int groups = tile == 64 && per_cu == 1 && n >= 4 ? 2 : 1;
      double cost = groups == 2 ? 0.3 + n * (elem_size == 4 ? 0.66 : 0.30) : per_cu == 1 ? n * alone : per_cu * n * shared;
      if (s > 1) cost += 2.5 + (double)s * M * N * 8 / 4e6;
      if (cost < best_cost) { best_cost = cost; best = {tile, s, groups}; }
    }
  }
  return best;
}
constexpr int kStep16 = 64, kStep32 = 32;   // contraction steps in LDS, 16-bit and fp32

template <typename T, bool AK, bool BKC> int launch_t(GemmArgs a, const Plan& p, hipStream_t stream) {
  constexpr int BK = sizeof(T) == 2 ? kStep16 : kStep32;
  const int tiles = ((a.M + p.tile - 1) / p.tile) * ((a.N + p.tile - 1) / p.tile);
  // at most what the CUs hold at once: two workgroups of 128 x 128 tiles or four of 64 x 64
  const dim3 grid(std::min((tiles + 7) / 8 * 8, p.tile == 128 ? 512 : 1024), p.splits);
  if constexpr (sizeof(T) == 2) {
    if (p.tile == 128) {
      hipLaunchKernelGGL((gemm_kernel<T, AK, BKC, 128, 128, BK, 1>), grid, dim3(kThreads), 0, stream, a);
      return hipGetLastError() == hipSuccess ? 0 : -3;
    }
  }
  if (p.groups == 2) hipLaunchKernelGGL((gemm_kernel<T, AK, BKC, 64, 64, BK, 2>), grid, dim3(2 * kThreads), 0, stream, a);
  else hipLaunchKernelGGL((gemm_kernel<T, AK, BKC, 64, 64, BK, 1>), grid, dim3(kThreads), 0, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace

int64_t gemm_workspace(int M, int N, int K, int elem_size, bool epilogue) {
  const Plan p = plan(M, N, K, !epilogue, elem_size);
  return p.splits > 1 ? (int64_t)p.splits * M * N * 4 : 0;
}

// the maximum is taken on the store: not for a contraction in ranges, nor for more tiles than there are slots
bool gemm_amax_ok(int M, int N, int K, int elem_size, int amax_from, int amax_to) {
  const Plan p = plan(M, N, K, true, elem_size);
  const int per_row = (amax_to - 1) / p.tile + 1 - amax_from / p.tile;
  return p.splits == 1 && (int64_t)((M + p.tile - 1) / p.tile) * per_row <= kAmaxBlocks;
}

int launch_gemm(GemmArgs a, bool a_kc, bool b_kc, int dtype, float* workspace, hipStream_t stream) {
  const int es = dtype == 0 ? 4 : 2, step = dtype == 0 ? kStep32 : kStep16;
  Plan p = plan(a.M, a.N, a.K, a.epilogue == kGemmPlain, es);
  a.k_per_split = ((a.K + p.splits - 1) / p.splits + step - 1) / step * step;
  p.splits = (a.K + a.k_per_split - 1) / a.k_per_split;   // rounding up may leave the last ones empty
  a.part = p.splits > 1 ? workspace : nullptr;
  const int rc = by_type(dtype, true, [&](auto t, auto) {
    using T = decltype(t);
    if (a_kc && b_kc) return launch_t<T, true, true>(a, p, stream);
    if (a_kc) return launch_t<T, true, false>(a, p, stream);
    if (!b_kc) return launch_t<T, false, false>(a, p, stream);
    return -2;
  });
  if (rc != 0 || a.part == nullptr) return rc;
  return launch_part_sum(a.part, p.splits, (int64_t)a.M * a.N, a.c, dtype, stream);
}

}  // namespace castle
