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
#include "castle_gelu.h"
#include "castle_waves.h"
#include <algorithm>
#include <cmath>
#include "castle_rows.h"

namespace castle {
namespace {

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
  static __device__ __forceinline__ int thread() { return G == 1 ? threadIdx.x : threadIdx.x % kThreads; }
  static __device__ __forceinline__ int row_of(int j) { return (thread() + j * kThreads) / VPR; }
  static __device__ __forceinline__ int col_of(int j) { return (thread() + j * kThreads) % VPR * V; }
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
    // (behind the end of the contraction the place of a next step may lie beyond 31 bits: it wraps, and is not read)
#pragma unroll
    for (int j = 0; j < N; ++j) at[j] = (int)((uint32_t)at[j] + (uint32_t)(KC ? G * BK : G * BK * ld));
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

constexpr int kStep16 = 64;   // contraction steps in LDS
// G: groups of four waves.  Two take alternate steps of the contraction for the same tile, each in LDS of its own, and are summed at
// the end: where the tiles leave a CU one workgroup, a second wave per SIMD works while the first waits for LDS and barrier.
// NORM: the rows of `a` are normalised between memory and LDS, one tile per workgroup.  Every workgroup reads its 64 rows once for
// their factors, with the first steps already on their way; that beats a launch in front of the product where the GPU is nearly empty.
template <typename T, bool AK, bool BKC, int BM, int BN, int BK, int G> constexpr int tile_elems() {
  return max2(G * 2 * (Operand<T, AK, BM, BK, G>::ELEMS + Operand<T, BKC, BN, BK, G>::ELEMS), BM * (BN + elem_traits<T>::vec16));
}
// workgroup (bx, by) of (gx, ...), in `smem` of tile_elems
template <typename T, bool AK, bool BKC, int BM, int BN, int BK, int G, bool NORM>
__device__ __forceinline__ void gemm_tiles(const GemmArgs& a, T* smem, int bx, int by, int gx) {
  constexpr int WM = BM / 64, WN = BN / 64;   // 32-wide pieces of a wave's quarter
  typedef Operand<T, AK, BM, BK, G> OpA;
  typedef Operand<T, BKC, BN, BK, G> OpB;
  constexpr int V = elem_traits<T>::vec16, LDC = BN + V;
  constexpr int kStage = 2 * (OpA::ELEMS + OpB::ELEMS);
  const int lane = lane_id(), wave = G == 1 ? wave_id() : wave_id() % 4, group = G == 1 ? 0 : wave_id() / 4, c = lane & 31, g = lane >> 5;
  // Workgroups go round the 8 XCDs, each with an L2 of its own: XCD x takes the x-th eighth of the tiles, so the rows of
  // `a` are read by one XCD, not by all (input gradient of 3000 rows x 1536 x 256: 13.5 -> 11.1 us).  A workgroup takes
  // several tiles where there are more than the CUs hold: the first steps of the next are requested before the
  // output of the last is written.
  const int tiles_n = (a.N + BN - 1) / BN, tiles = (a.M + BM - 1) / BM * tiles_n;
  const int share = (tiles + 7) / 8, first = bx % 8 * share, last = min(tiles, first + share);
  const int wm = wave / 2 * (BM / 2), wn = wave % 2 * (BN / 2);
  const int k0 = by * a.k_per_split, k_end = min(a.K, k0 + a.k_per_split);
  const int steps = ((k_end - k0 + BK - 1) / BK + G - 1) / G;   // of a group: its steps are G BK apart
  T* const stage = smem + group * kStage;
  const T *pa = static_cast<const T*>(a.a), *pb = static_cast<const T*>(a.b);
  OpA ra;
  OpB rb;
  acc_t acc[WM][WN];   // [n rows, m lanes]
  int tile = first + bx / 8;
  auto request = [&]() __attribute__((always_inline)) {
    ra.start((int)a.lda, tile / tiles_n * BM, a.M, k0 + group * BK);
    rb.start((int)a.ldb, tile % tiles_n * BN, a.N, k0 + group * BK);
#pragma unroll
    for (int p = 0; p < 2; ++p) {   // (a step beyond the end loads zeros)
      ra.load(p, pa, (int)a.lda, k0 + (p * G + group) * BK, k_end);
      rb.load(p, pb, (int)a.ldb, k0 + (p * G + group) * BK, k_end);
    }
  };
  __shared__ __attribute__((aligned(16))) float s_norm[NORM ? kNormBytes / (int)sizeof(T) : 4], s_factor[NORM ? BM : 1];
  const int m_first = tile / tiles_n * BM;
  const bool norm_keeps = NORM && a.h != nullptr && tile % tiles_n == 0;   // (the first column of tiles stores what all of them form)
  auto step = [&](auto parity, int it) __attribute__((always_inline)) {
    constexpr int p = decltype(parity)::value;
    T* la = stage + p * (OpA::ELEMS + OpB::ELEMS);
    T* lb = la + OpA::ELEMS;
    if constexpr (NORM) {
      const int k = k0 + (it * G + group) * BK;
#pragma unroll
      for (int j = 0; j < OpA::N; ++j) {
        const int row = OpA::row_of(j), col = k + OpA::col_of(j);
        typedef vec<float, V> vf;
        if (col < a.K) {
          ra.r[p][j] = __builtin_convertvector(__builtin_convertvector(ra.r[p][j], vf) * s_factor[row] * *reinterpret_cast<const vf*>(s_norm + col), vec<T, V>);
          if (norm_keeps && m_first + row < a.M) *reinterpret_cast<vec<T, V>*>(static_cast<T*>(a.h) + (int64_t)(m_first + row) * a.K + col) = ra.r[p][j];
        }
      }
    }
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
  if (a.amax != nullptr && bx == 0) {
    for (int i = (a.M + BM - 1) / BM * amax_tiles + threadIdx.x; i < kAmaxBlocks; i += kThreads * G) a.amax[i] = 0.f;
    if (threadIdx.x == 0 && a.amax_status != nullptr) *a.amax_status = 0;
  }
  if (tile < last) request();
  if constexpr (NORM) {
    if (tile < last) {
      constexpr int LPR = kThreads * G / BM;   // lanes of a row
      static_assert(64 % LPR == 0, "a row in one wave");
      typedef vec<float, V> vf;
      const int row = threadIdx.x / LPR, sub = threadIdx.x % LPR;
      const T* x = pa + (int64_t)min(m_first + row, a.M - 1) * a.lda;
      // summed in the order of the norm by itself (16, 32 or 64 lanes to a row, added in pairs), PER of whose lanes a lane here stands for:
      // the layer gives the same bits by either way
      const int pieces = a.K / V;
      auto sum_of = [&](auto per, int lanes) __attribute__((always_inline)) {
        constexpr int PER = decltype(per)::value;
        float sum[PER];
#pragma unroll
        for (int v = 0; v < PER; ++v) sum[v] = 0.f;
        for (int first = 0; first < pieces; first += lanes) {
#pragma unroll
          for (int v = 0; v < PER; ++v) {
            const int i = first + sub * PER + v;
            const vf f = __builtin_convertvector(*reinterpret_cast<const vec<T, V>*>(x + (i < pieces ? i : 0) * V), vf);
#pragma unroll
            for (int e = 0; e < V; ++e) {
              const float g = i < pieces ? f[e] : 0.f;
              sum[v] = __builtin_fmaf(g, g, sum[v]);
            }
          }
        }
#pragma unroll
        for (int o = 1; o < PER; o <<= 1)
#pragma unroll
          for (int v = 0; v < PER; v += 2 * o) sum[v] += sum[v + o];
        return sum[0];
      };
      float ssq = pieces <= 16 ? sum_of(std::integral_constant<int, 16 / LPR>(), 16)
                               : pieces <= 32 ? sum_of(std::integral_constant<int, 32 / LPR>(), 32) : sum_of(std::integral_constant<int, 64 / LPR>(), 64);
      for (int i = threadIdx.x; i < a.K; i += kThreads * G) s_norm[i] = (float)static_cast<const T*>(a.norm_w)[i];
#pragma unroll
      for (int o = 1; o < LPR; o <<= 1) ssq += __shfl_xor(ssq, o);
      const float r = 1.f / sqrtf(ssq / (float)a.K + a.eps);
      if (sub == 0) {
        s_factor[row] = r;
        if (norm_keeps && a.rstd != nullptr && m_first + row < a.M) a.rstd[m_first + row] = r;
      }
      __syncthreads();
    }
  }
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
      static_assert(kThreads * WM * WN * 64 <= (int)sizeof(T) * tile_elems<T, AK, BKC, BM, BN, BK, G>(), "one group's sums");
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
    tile += gx / 8;
    if (tile < last) request();
    if (a.part != nullptr) {   // partial product of this range of the contraction
      float* part = a.part + (int64_t)by * a.M * a.N;
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
      if (lane == 0) s_most[G == 1 ? wave : wave_id()] = most;
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
template <typename T, bool AK, bool BKC, int BM, int BN, int BK, int G, bool NORM = false>
__global__ __launch_bounds__(kThreads * G, BM == 128 ? 2 : 4) void gemm_kernel(GemmArgs a) {
  __shared__ __attribute__((aligned(16))) T smem[tile_elems<T, AK, BKC, BM, BN, BK, G>()];
  gemm_tiles<T, AK, BKC, BM, BN, BK, G, NORM>(a, smem, blockIdx.x, blockIdx.y, gridDim.x);
}
// Both gradients of a projection, which read the same dy and nothing of each other, in one launch: workgroups of the weight gradient
// (w.k_per_split rows of the contraction each), then those of the input gradient.
// Each by itself is bound by its start, trips to memory and CUs that stay idle; together they fill them (3000 rows 256 -> 1536, us: 16.8 and 11.4, both 19.0; the rule and
// more figures at grads_plan).  Tiles of 64 x 64 for both, by one or two groups: larger ones do not leave a CU room for a workgroup of the other.
template <typename T, int G> __global__ __launch_bounds__(kThreads * G, 4) void grads_kernel(GradsArgs p) {
  constexpr int kElems = max2(tile_elems<T, false, false, 64, 64, kStep16, G>(), tile_elems<T, true, false, 64, 64, kStep16, G>());
  __shared__ __attribute__((aligned(16))) T smem[kElems];
  int b = blockIdx.x;
  if (b < p.w_groups) {
    gemm_tiles<T, false, false, 64, 64, kStep16, G, false>(p.w, smem, b % p.w_row, b / p.w_row, p.w_row);
  } else {
    b -= p.w_groups;
    gemm_tiles<T, true, false, 64, 64, kStep16, G, false>(p.x, smem, b % p.x_row, b / p.x_row, p.x_row);
  }
}

// ---- large products of 16-bit operands -----------------------------------------------------------------------------------------
// 256 x 128 or 256 x 256 of the output per workgroup of eight waves, one workgroup per CU.  What bounds a step of the contraction (64) is
// the way from L2 into the CU, about 29 bytes a clock (256 x 128: 48 KB in 0.70 us with the products left out, 0.55 us for the products
// without it, 0.75 together), so larger tiles, which read less for each product: 0.75 ... 1.0 us a step for 256 x 128, 1.4 ... 1.6 for
// 256 x 256, where 128 x 128 tiles of gemm_kernel take 0.6.  The steps go straight from memory to LDS, into three buffers (two of 256 x
// 256), the next ones on their way while one is multiplied, over the end of a tile too; the stores of a tile are not waited for.
// 16384 rows, us, gemm_kernel / here / the library (outputs not in a cache): 512 -> 2048 59 / 43 / 45, with gelu 80 / 64 / 76; 512 -> 3072
// 86 / 61 / 66; 512 -> 512 18 / 16 / 20; 8192 rows of 512 -> 3072 46 / 36 / 51, 3072 -> 512 49 / 44 / 39.
// 16-byte pieces go to LDS in the order of the lanes, so rows cannot be padded: a piece takes another place in its row instead, such that
// the lanes of a read spread over all banks (contraction-contiguous: piece p of row r at p ^ (r / 2 % 8); else the pieces of row k
// at p ^ 4 (k % 4)).
constexpr int kWideM = 256, kWideK = 64, kWideThreads = 512;
template <int BN> struct Wide {
  static constexpr int kStages = BN == 256 ? 2 : 3;
  static constexpr int kStage = (kWideM + BN) * kWideK * 2;   // bytes
  static constexpr int kLoads = kStage / 1024 / (kWideThreads / 64);   // of a wave and step, 1 KB each
  // where a wave turns 32 rows of its outputs, 4 KB: behind the buffers if there is room, else in the one of the last step
  static constexpr bool kOwnTurn = BN == 256;
  static constexpr int kLds = kStages * kStage + (kOwnTurn ? 4096 * kWideThreads / 64 : 4 * kWideThreads / 64);   // and a maximum of each wave
};
template <typename T, bool KC, int FREE> struct WideOperand {
  static constexpr int N = FREE / 64;   // loads of a wave
  const T* at;
  uint32_t off[N];   // bytes
  __device__ __forceinline__ void start(const T* p, int64_t ld, int free0, int free_end, int k0) {
    const int lane = lane_id(), first = wave_id() * N;
    at = KC ? p + free0 * ld + k0 : p + k0 * ld + free0;
#pragma unroll
    for (int q = 0; q < N; ++q) {
      if constexpr (KC) {
        const int row = 8 * (first + q) + (lane >> 3), piece = (lane & 7) ^ (row >> 1 & 7);
        off[q] = 2 * (uint32_t)((int)ld * min(row, free_end - 1 - free0) + 8 * piece);
      } else {
        constexpr int PIECES = FREE / 8, ROWS = 64 / PIECES;
        const int k = ROWS * (first + q) + lane / PIECES, piece = lane % PIECES ^ 4 * (k & 3);
        off[q] = 2 * (uint32_t)(k * (int)ld + (free0 + 8 * piece < free_end ? 8 * piece : 0));
      }
    }
  }
  __device__ __forceinline__ void load(int64_t ld, uint32_t lds) {
#pragma unroll
    for (int q = 0; q < N; ++q) load_to_lds(at, off[q], lds + 1024 * (wave_id() * N + q));
    at += KC ? kWideK : kWideK * ld;
  }
  // operand fragments of the wave's 32 W columns from free0, 16 contraction steps from 16 s
  template <int W> static __device__ __forceinline__ void read(const T* lds, frag<T> (&f)[W], int free0, int s, int c, int g) {
    if constexpr (KC) {
      const T* p = lds + (free0 + c) * kWideK + 8 * ((2 * s + g) ^ (c >> 1 & 7));
#pragma unroll
      for (int i = 0; i < W; ++i) f[i] = *reinterpret_cast<const frag<T>*>(p + 32 * kWideK * i);
    } else {
      const int lp = c & 15, k = 16 * s + 8 * g + (lp >> 2);
#pragma unroll
      for (int i = 0; i < W; ++i) {
        const T* p = lds + k * FREE + 32 * ((free0 / 32 + i) ^ (lp >> 2)) + 16 * (c >> 4) + 4 * (lp & 3);
        const vec<T, 4> lo = lds_tr4<T>(p), hi = lds_tr4<T>(p + 4 * FREE);
#pragma unroll
        for (int e = 0; e < 4; ++e) { f[i][e] = lo[e]; f[i][4 + e] = hi[e]; }
      }
    }
  }
};
extern __shared__ __attribute__((aligned(16))) unsigned char castle_wide[];

// FUSED: with gelu or its derivative on the store (kernels of their own: the code of a plain store stays short)
template <typename T, bool AK, bool BKC, int BN, bool FUSED> __global__ __launch_bounds__(kWideThreads, 2) void gemm_wide_kernel(GemmArgs a) {
  typedef Wide<BN> W;
  constexpr int WN = BN / 64;   // 32-wide pieces of a wave
  typedef WideOperand<T, AK, kWideM> OpA;
  typedef WideOperand<T, BKC, BN> OpB;
  typedef vec<T, 8> vt;
  typedef vec<float, 8> vf;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  // Tiles in the order of an XCD's L2: all rows of eight columns of tiles (2048 output columns), then those of the next.
  constexpr int kBand = 2048 / BN;
  const int tiles_m = (a.M + kWideM - 1) / kWideM, tiles_n = (a.N + BN - 1) / BN, tiles = tiles_m * tiles_n;
  auto place = [&](int t, int& m0, int& n0) __attribute__((always_inline)) {
    const int band = t / (tiles_m * kBand), rest = t - band * tiles_m * kBand, width = min(kBand, tiles_n - band * kBand);
    m0 = rest / width * kWideM;
    n0 = (band * kBand + rest % width) * BN;
  };
  const int share = (tiles + 7) / 8, first = blockIdx.x % 8 * share, last = min(tiles, first + share), stride = gridDim.x / 8;
  const int wm = wave / 2 * 64, wn = wave % 2 * (BN / 2);
  const int k0 = blockIdx.y * a.k_per_split, steps = (min(a.K, k0 + a.k_per_split) - k0) / kWideK;
  const int amax_tile = a.amax_from / BN, amax_tiles = (a.amax_to - 1) / BN + 1 - amax_tile;   // of a row of tiles
  if (a.amax != nullptr && blockIdx.x == 0) {
    for (int i = (a.M + kWideM - 1) / kWideM * amax_tiles + threadIdx.x; i < kAmaxBlocks; i += kWideThreads) a.amax[i] = 0.f;
    if (threadIdx.x == 0 && a.amax_status != nullptr) *a.amax_status = 0;
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)castle_wide;
  int tile = first + blockIdx.x / 8;
  if (tile >= last) return;
  // the step that is requested next runs ahead of the one that is multiplied, into the next tile
  OpA ra;
  OpB rb;
  int next_tile = tile, next_step = 0, ahead = 0;   // ahead: steps requested and not waited for
  auto start = [&]() __attribute__((always_inline)) {
    int m0, n0;
    place(next_tile, m0, n0);
    ra.start(static_cast<const T*>(a.a), a.lda, m0, a.M, k0);
    rb.start(static_cast<const T*>(a.b), a.ldb, n0, a.N, k0);
  };
  auto request = [&](int buffer) __attribute__((always_inline)) {
    if (next_tile >= last) return;
    ++ahead;
    ra.load(a.lda, lds0 + buffer);
    rb.load(a.ldb, lds0 + buffer + kWideM * kWideK * 2);
    if (++next_step == steps) {
      next_step = 0;
      next_tile += stride;
      if (next_tile < last) start();
    }
  };
  start();
  request(0);
  request(W::kStage);
  if constexpr (W::kStages == 3) request(2 * W::kStage);
  // The step behind the current one is in LDS, from every wave, and all have read the current one.  Waits are for all but the last so many
  // requests; the stores of a tile that lies inside the output are counted (STORES more), so they are not waited for.
  constexpr int STORES = 4 * WN;
  int stores = 0;   // 1: the stores of the tile before are behind the pieces that are waited for, 2: as many again
  auto arrive = [&]() __attribute__((always_inline)) {
    auto wait = [&](auto n) __attribute__((always_inline)) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(decltype(n)::value) : "memory");
    };
    const int newer = ahead - 1;   // steps
    if (newer > 1) wait(std::integral_constant<int, 2 * W::kLoads>());
    else if (newer == 1) {
      if (stores == 2) wait(std::integral_constant<int, W::kLoads + 2 * STORES>());
      else if (stores == 1) wait(std::integral_constant<int, W::kLoads + STORES>());
      else wait(std::integral_constant<int, W::kLoads>());
    } else {
      if (stores == 2) wait(std::integral_constant<int, 2 * STORES>());
      else if (stores == 1) wait(std::integral_constant<int, STORES>());
      else wait(std::integral_constant<int, 0>());
    }
    stores = 0;
    --ahead;
  };
  int buffer = 0;
  frag<T> fa[2][2], fb[2][WN];
  auto read = [&](int slot, int s) __attribute__((always_inline)) {
    const T* la = reinterpret_cast<const T*>(castle_wide + buffer);
    OpA::read(la, fa[slot], wm, s, c, g);
    OpB::read(la + kWideM * kWideK, fb[slot], wn, s, c, g);
    __builtin_amdgcn_sched_barrier(0);   // these reads, then the products of the fragments before
  };
  arrive();
  read(0, 0);
  while (tile < last) {
    int m0, n0;
    place(tile, m0, n0);
    acc_t acc[2][WN];   // [n rows, m lanes]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < WN; ++j) zero(acc[i][j]);
    auto multiply = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j) mma(acc[i][j], fb[slot][j], fa[slot][i]);
    };
    int done = 0;   // buffer of the step that ends
    for (int it = 0; it < steps; ++it) {
#pragma unroll
      for (int s = 0; s < kWideK / 16 - 1; ++s) {
        read(1 - s % 2, s + 1);
        multiply(s % 2);
      }
      arrive();
      done = buffer;
      buffer = buffer == (W::kStages - 1) * W::kStage ? 0 : buffer + W::kStage;
      if (it + 1 < steps) request(done);
      read(0, 0);   // (behind the last step of all: what is there, for nothing)
      multiply(1);
    }
    asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");   // the loop may end right behind a product
    __builtin_amdgcn_sched_barrier(0);
    tile += stride;
    const bool inside = m0 + kWideM <= a.M && n0 + BN <= a.N;
    if (a.part != nullptr) {   // partial product of this range of the contraction
      request(done);
      float* part = a.part + (int64_t)blockIdx.y * a.M * a.N;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < WN; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int m = m0 + wm + 32 * i + c, n = n0 + wn + 32 * j + 8 * q + 4 * g;
            if (m < a.M && n < a.N) *reinterpret_cast<vec<float, 4>*>(part + (int64_t)m * a.N + n) = pack4<float>(acc[i][j], q);
          }
      if (inside) stores = 2;
      continue;
    }
    // to whole rows through the buffer of the last step, each wave in the part that it fills next; pieces placed as above
    static_assert(OpA::N * 1024 == 32 * 64 * 2, "32 rows of each wave");
    if constexpr (W::kOwnTurn) request(done);
    T* out = reinterpret_cast<T*>(castle_wide + (W::kOwnTurn ? W::kStages * W::kStage : done) + wave * 4096);
    float most = 0.f;
    // the second operand of the slope is on its way a piece ahead
    vt u[2][4];
    auto fetch = [&](int h) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 32 * (h % 2) + 8 * r + (lane >> 3), n = n0 + wn + 64 * (h / 2) + 8 * (lane & 7);
        u[h % 2][r] = *reinterpret_cast<const vt*>(static_cast<const T*>(a.aux) + (int64_t)min(m, a.M - 1) * a.ldc + (n < a.N ? n : 0));
      }
    };
    const bool slope = FUSED && a.epilogue == kGemmGeluSlope, gelu_too = FUSED && a.epilogue == kGemmGelu;
    if (slope) fetch(0);
#pragma unroll
    for (int h = 0; h < WN; ++h) {   // 32 x 64 of the wave's part
      const int i = h % 2, half = h / 2;
      if (slope && h + 1 < WN) fetch(h + 1);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) st4<T>(out + c * 64 + 8 * ((4 * j + q) ^ (c >> 1 & 7)) + 4 * g, pack4<T>(acc[i][2 * half + j], q));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 8 * r + (lane >> 3), m = m0 + wm + 32 * i + row, n = n0 + wn + 64 * half + 8 * (lane & 7);
        vt x = *reinterpret_cast<const vt*>(out + row * 64 + 8 * ((lane & 7) ^ (row >> 1 & 7)));
        if (m >= a.M || n >= a.N) continue;
        const int64_t at = (int64_t)m * a.ldc + n;
        if (slope) {
          vf f = __builtin_convertvector(x, vf);
          const vf v = __builtin_convertvector(u[i][r], vf);
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] *= gelu_slope<T>(v[e]);
          x = __builtin_convertvector(f, vt);
        }
        *reinterpret_cast<vt*>(static_cast<T*>(a.c) + at) = x;
        if (a.amax != nullptr && n >= a.amax_from && n < a.amax_to) {
          const vf f = __builtin_convertvector(x, vf);
#pragma unroll
          for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(f[e]));   // fmaxf drops NaNs
        }
        if (gelu_too) {
          vf f = __builtin_convertvector(x, vf);
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] = gelu<T>(f[e]);
          *reinterpret_cast<vt*>(static_cast<T*>(a.aux) + at) = __builtin_convertvector(f, vt);
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (!W::kOwnTurn) request(done);
    if (inside) stores = gelu_too ? 2 : 1;
    const int slot = n0 / BN - amax_tile;
    if (a.amax != nullptr && slot >= 0 && slot < amax_tiles) {
      constexpr int kApart = W::kOwnTurn ? 1024 : 1;   // in the wave's own part
      float* s_most = reinterpret_cast<float*>(castle_wide + W::kStages * W::kStage);
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) most = fmaxf(most, __shfl_xor(most, o));
      if (lane == 0) s_most[wave * kApart] = most;
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (threadIdx.x == 0) {
#pragma unroll
        for (int w = 1; w < kWideThreads / 64; ++w) most = fmaxf(most, s_most[w * kApart]);
        a.amax[m0 / kWideM * amax_tiles + slot] = fminf(most, 3.0e38f);   // an infinite value counts as the largest finite one
      }
    }
  }
}

// Tile, number of ranges of the contraction and groups of a workgroup, from what a launch takes (us): a start (2.3 for tiles of 64 and 128 rows, where
// gelu or its derivative rides on the store within the end of a tile), and for each tile of the fullest CU so much a step and at its end, more at the end where
// gelu or its derivative rides on the store.  A second group takes a step of a workgroup of 64 x 64 that has a CU to itself from 0.42 to 0.36,
// for 0.3 at the end, and pays from eight steps on (3000 rows of 1536 -> 256 12.7 with one, 9.9 with two, 1504 rows of 256 -> 512 5.3 and 6.1);
// at two workgroups a CU it gains where the contraction is long (3000 rows of 3072 -> 512 29 / 26, of 512 -> 512
// level), behind from three on.  A split adds a second launch, 2.5, and its partial results, written and read, and tiles of 256 rows another start.
// Weight gradient of 3000 rows, 1536 x 256 out: 22.6 in one range, 13.7 in two of two groups; 3008 rows 512 -> 2048 17.6 on 64 x 64, 16.6 on 128 x 128, 14.2 on
// 256 x 128; 4096 rows 512 -> 3072 31.8, 26.2, 24.9 and 21.8 on 256 x 256; 8184 rows 64 -> 4096 20.0, 18.6, 15.8 and 15.3.  Over 2500 products of 96 ... 65536
// rows, outputs of 64 ... 4096 columns and contractions of 64 ... 8184, in all layouts, each timed with every tile and up to 16 ranges, what this picks takes 1.5 %
// more than the best of them on average.
struct Plan {
  int tile, splits, groups;   // tile: 32 (fp32), 64, 128, or columns of a tile of 256 rows + 256; groups: of four waves
  int waves = 0;    // fp32
  float cost = 0;   // us, roughly
  int rows() const { return std::min(tile, kWideM); }
  int columns() const { return tile > kWideM ? tile - kWideM : tile; }
  int tiles(int M, int N) const { return ((M + rows() - 1) / rows()) * ((N + columns() - 1) / columns()); }
};
// workgroups of the fullest CU: tiles go to eight XCDs of 32 CUs each, so one of them may have work for 33 (weight gradient of 8184 rows, 640 x 320: 50 tiles in
// five ranges 21.6 us, in four 16.9)
int64_t on_a_cu(int64_t tiles, int splits) { return ((tiles + 7) / 8 * splits + 31) / 32; }
// fp32 (castle_gemm32.hip): tiles of 64 x 64 by one, two or four waves and of 32 x 32 by four or eight, `held` workgroups to a CU at once.  From what a launch takes (us): a
// start, and for the workgroups of the fullest CU, so many at a time, so much for a wave's 32 steps and at the end (one by itself, and all of them); or so much for a MB that
// the tiles read, and between the two where they are level; a split adds the sum of its ranges.  Fitted to 190000 timings of 9358 products of 16 ... 23000 rows, outputs of
// 32 ... 4096 columns and contractions of 16 ... 23000, in all layouts.  What it picks takes 2 % more than the best of them on average, 8 % in one of ten, and 0.74 of what the
// library takes, 1.02 in one of ten.
Plan plan32(int M, int N, int K, bool plain) {
  struct Kind { int tile, waves, held; float start, step, end, steps, ends, split, split_mb, read; };
  constexpr Kind kinds[5] = {{64, 1, 8, 6.03f, 1.47f, 0.219f, 1.63f, 6.29f, 1.65f, 0.201f, 0.101f},
                             {64, 2, 4, 4.28f, 1.51f, 1.62f, 3.33f, 3.03f, 1.72f, 0.218f, 0},
                             {64, 4, 2, 4.07f, 1.61f, 1.58f, 2.51f, 2.33f, 1.93f, 0.213f, 0.097f},
                             {32, 8, 2, 4.22f, 0.99f, 0, 1.61f, 0.304f, 2.03f, 0.25f, 0.078f},
                             {32, 4, 4, 4.15f, 0.752f, 0.047f, 1.52f, 0.771f, 2.06f, 0.209f, 0.071f}};
  Plan best = {64, 1, 1, 4};
  float best_cost = 1e30f;
  const auto tiles_of = [&](int tile) { return (int)std::min<int64_t>((int64_t)((M + tile - 1) / tile) * ((N + tile - 1) / tile), 1 << 26); };
  const int tiles64 = tiles_of(64), tiles32 = tiles_of(32);
  const float mb = 8e-6f * M * N;
  for (const int s : {1, 2, 3, 4, 6, 8, 12, 16}) {   // (a call looks at all this three times: no divisions and roots that can be spared)
    if (s > 1 && (!plain || s > (K + 31) / 32 || tiles64 * s > 1024)) break;
    const int stages = ((K + s - 1) / s + 31) / 32;
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      const Kind& kind = kinds[k];
      const int tiles = kind.tile == 64 ? tiles64 : tiles32, per_cu = (int)on_a_cu(tiles, s), rounds = (stages + kind.waves - 1) / kind.waves;
      const int rest = per_cu % kind.held;
      const float full = rest > 1 ? (rest - 1.f) / (kind.held - 1) : 0.f;   // of the way from one by itself to all of them
      float work = per_cu / kind.held * (rounds * kind.steps + kind.ends);
      if (rest > 0) work += rounds * (kind.step + full * (kind.steps - kind.step)) + kind.end + full * (kind.ends - kind.end);
      const float fixed = kind.start + (s > 1 ? kind.split + s * mb * kind.split_mb : 0.f);
      if (fixed + work >= best_cost) continue;
      const float read = 8e-6f * tiles * K * kind.tile * kind.read, w2 = work * work, r2 = read * read, cost = fixed + std::sqrt(std::sqrt(w2 * w2 + r2 * r2));
      if (cost < best_cost) { best_cost = cost; best = {kind.tile, s, std::max(1, kind.waves / 4), kind.waves, cost}; }
    }
  }
  return best;
}
Plan plan(int M, int N, int K, bool plain, int elem_size) {
  if (elem_size == 4) return plan32(M, N, K, plain);
  Plan best = {64, 1, 1};
  double best_cost = 1e30;
  auto take = [&](double cost, const Plan& p) {
    if (cost < best_cost) { best_cost = cost; best = p; best.cost = (float)cost; }
  };
  // Two tensors that no cache holds: stores of single lines cost more (gelu of 65536 rows 64 -> 1536 on 64 x 64 123, on 256 x 256 94), and 256 x 256 where rows do not
  // start with lines (33000 rows 64 -> 3064 192, 256 x 128 103, 64 x 64 150).
  const bool far = !plain && 4.0 * M * N > 2.5e8;
  for (int tile = 64; tile <= 128; tile += 64) {
    const double alone = tile == 64 ? 0.42 : 0.85, shared = tile == 64 ? 0.29 : 0.6;
    const double fused = plain ? 0 : tile == 128 ? 2.6 : far ? 1 : 0.5;
    const int64_t tiles = (int64_t)((M + tile - 1) / tile) * ((N + tile - 1) / tile);
    const int steps = (K + kStep16 - 1) / kStep16;
    for (int s = 1; s <= (plain ? std::min(16, (steps + 1) / 2) : 1); ++s) {
      const int64_t per_cu = on_a_cu(tiles, s), n = (steps + s - 1) / s;
      const double end = tile == 64 ? 0.25 : s > 1 ? 1 : 2.3;   // (partial results do not go through LDS)
      const int groups = tile == 64 && (per_cu == 1 ? n >= 8 : s == 1 && per_cu == 2 && n >= 12) ? 2 : 1;
      double cost = groups == 2 ? 0.3 + n * (per_cu == 1 ? 0.36 : 0.55) : per_cu == 1 ? n * alone + end : per_cu * (n * shared + end);
      if (s > 1) cost += 2.5 + (double)s * M * N * 8 / 4e6;
      take((plain ? 2.3 : 0) + cost + (per_cu == 1 ? 2 : per_cu) * fused, {tile, s, groups});
    }
  }
  if (K % kWideK == 0) {
    for (int columns = 128; columns <= 256; columns += 128) {
      const double start = plain ? 3.5 : columns == 128 ? 1.6 : 2.6, end = columns == 128 ? (plain ? 1.8 : 8.8) : plain ? 4 : far && N % 64 != 0 ? 24.5 : 16.5;
      const int64_t tiles = (int64_t)((M + kWideM - 1) / kWideM) * ((N + columns - 1) / columns);
      const int steps = K / kWideK;
      for (int s = 1; s <= (plain ? std::min(16, std::max(1, steps / 4)) : 1); ++s) {
        const int64_t per_cu = on_a_cu(tiles, s), n = (steps + s - 1) / s;
        const double busy = std::min(1., tiles * s / 256.), step = columns == 128 ? 0.75 + 0.27 * busy : 1.2 + 0.36 * busy;
        take(start + per_cu * (n * step + end) + (s > 1 ? 4.8 + (double)s * M * N * 8 / 6e6 : 0), {kWideM + columns, s, 1});
      }
    }
  }
  return best;
}
template <typename T, bool AK, bool BKC, int BN, bool FUSED> int launch_wide(const GemmArgs& a, const Plan& p, hipStream_t stream) {
  static PerDeviceOnce once;
  bool& configured = once.flag();
  if (!configured) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wide_kernel<T, AK, BKC, BN, FUSED>), hipFuncAttributeMaxDynamicSharedMemorySize, Wide<BN>::kLds) != hipSuccess) return -3;
    configured = true;
  }
  hipLaunchKernelGGL((gemm_wide_kernel<T, AK, BKC, BN, FUSED>), dim3(std::min((p.tiles(a.M, a.N) + 7) / 8 * 8, 256), p.splits), dim3(kWideThreads), Wide<BN>::kLds, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

template <typename T, bool AK, bool BKC> int launch_t(GemmArgs a, const Plan& p, hipStream_t stream) {
  constexpr int BK = kStep16;
  const int tiles = p.tiles(a.M, a.N);
  // at most what the CUs hold at once: two workgroups of 128 x 128 tiles or four of 64 x 64
  const dim3 grid(std::min((tiles + 7) / 8 * 8, p.tile == 128 ? 512 : 1024), p.splits);
  if (p.tile > kWideM) {
    const bool plain = a.epilogue == kGemmPlain;
    if (p.columns() == 128) return plain ? launch_wide<T, AK, BKC, 128, false>(a, p, stream) : launch_wide<T, AK, BKC, 128, true>(a, p, stream);
    return plain ? launch_wide<T, AK, BKC, 256, false>(a, p, stream) : launch_wide<T, AK, BKC, 256, true>(a, p, stream);
  }
  if (p.tile == 128) {
    hipLaunchKernelGGL((gemm_kernel<T, AK, BKC, 128, 128, BK, 1>), grid, dim3(kThreads), 0, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -3;
  }
  // (both operands contraction-strided at two workgroups a CU: one group, weight gradients of 1000 rows 512 x 3072 13.2 us and with two 14.2, of 3000 30.4 / 32.1)
  if (p.groups == 2 && (AK || on_a_cu(tiles, p.splits) == 1)) hipLaunchKernelGGL((gemm_kernel<T, AK, BKC, 64, 64, BK, 2>), grid, dim3(2 * kThreads), 0, stream, a);
  else hipLaunchKernelGGL((gemm_kernel<T, AK, BKC, 64, 64, BK, 1>), grid, dim3(kThreads), 0, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace

int64_t gemm_workspace(int M, int N, int K, int elem_size, bool epilogue) {
  const Plan p = plan(M, N, K, !epilogue, elem_size);
  return p.splits > 1 ? (int64_t)p.splits * M * N * 4 : 0;
}

void gemm_plan(int M, int N, int K, int elem_size, bool epilogue, int (&out)[4]) {
  const Plan p = plan(M, N, K, !epilogue, elem_size);
  out[0] = p.rows(); out[1] = p.columns(); out[2] = p.splits; out[3] = p.groups;
}

// the maximum is taken on the store: not for a contraction in ranges, nor for more tiles than there are slots
bool gemm_amax_ok(int M, int N, int K, int elem_size, int amax_from, int amax_to) {
  const Plan p = plan(M, N, K, true, elem_size);
  const int per_row = (amax_to - 1) / p.columns() + 1 - amax_from / p.columns();
  return p.splits == 1 && (int64_t)((M + p.rows() - 1) / p.rows()) * per_row <= kAmaxBlocks;
}

// One tile per workgroup and a CU for each (or for four of 32 rows), so that a row is read for its factor where it costs nothing else; tile and groups of the product
// by itself, for the same bits.
bool gemm_norm_ok(int M, int N, int K, int elem_size) {
  if ((int64_t)K * elem_size > kNormBytes) return false;
  const Plan p = plan(M, N, K, true, elem_size);
  return p.tile <= 64 && p.splits == 1 && p.tiles(M, N) * p.tile * p.tile <= 256 * 64 * 64 && (elem_size == 2 || p.waves >= 4);
}

int launch_gemm(GemmArgs a, bool a_kc, bool b_kc, int dtype, float* workspace, hipStream_t stream) {
  const int es = dtype == 0 ? 4 : 2, step = dtype == 0 ? 32 : kStep16;
  Plan p = plan(a.M, a.N, a.K, a.epilogue == kGemmPlain || a.amax != nullptr, es);   // (the slots of the maxima follow from the plain plan)
  a.k_per_split = ((a.K + p.splits - 1) / p.splits + step - 1) / step * step;
  p.splits = (a.K + a.k_per_split - 1) / a.k_per_split;   // rounding up may leave the last ones empty
  a.part = p.splits > 1 ? workspace : nullptr;
  const int rc = dtype == 0 ? launch_gemm32(a, a_kc, b_kc, p.tile, p.splits, p.waves, stream) : by_type16(dtype, true, [&](auto t, auto) {
    using T = decltype(t);
    if (a.norm_w != nullptr) {
      const dim3 grid((p.tiles(a.M, a.N) + 7) / 8 * 8);
      if (p.groups == 2) hipLaunchKernelGGL((gemm_kernel<T, true, true, 64, 64, kStep16, 2, true>), grid, dim3(2 * kThreads), 0, stream, a);
      else hipLaunchKernelGGL((gemm_kernel<T, true, true, 64, 64, kStep16, 1, true>), grid, dim3(kThreads), 0, stream, a);
      return hipGetLastError() == hipSuccess ? 0 : -3;
    }
    if (a_kc && b_kc) return launch_t<T, true, true>(a, p, stream);
    if (a_kc) return launch_t<T, true, false>(a, p, stream);
    if (!b_kc) return launch_t<T, false, false>(a, p, stream);
    return -2;
  });
  if (rc != 0 || a.part == nullptr) return rc;
  return launch_part_sum(a.part, p.splits, (int64_t)a.M * a.N, a.c, dtype, stream);
}

// Both gradients of a projection in one launch, y = x w^T with R rows, N outputs, K inputs.  They are launches of a few us that leave CUs idle, each with a start,
// a trip to memory and a last wave of its own.  What one launch of both takes (us): a start, and the 4-norm of the longest workgroup by itself, of the steps and ends
// of all workgroups spread over the CUs, and of what the tiles read; ranges of a contraction add the launch that sums them and their partial results.  Fitted to 49000
// timings of 2904 projections of 16 ... 8192 rows, widths of 64 ... 6144 and up to 40 GFLOP.  One launch is taken where this is clearly less than the plans of the two
// by themselves, in four of five of those, 1.4 times as fast there in 16 bit and 1.3 in fp32 (all of them: 1.32 and 1.2; slower by more than 4 % in 0 and 0.4 %).  Two against
// one, us: bf16 3000 rows 256 -> 1536 25.1 / 19.0, 256 -> 256 13.6 / 10.0, 199 rows 384 -> 384 9.9 / 6.0, fp32 256 rows 512 -> 3072 28.5 / 24.6, 512 -> 512 10.6 / 8.4;
// bf16 977 rows 768 -> 4608, where one of the two has larger tiles, 42.3 / 52.6.
GradsPlan grads_plan(int R, int N, int K, int elem_size, int epilogue, bool amax) {
  struct Kind { int tile, waves, turns; float start, alone, shared, end, ends, split, split_mb, read; };   // turns: steps at a time
  constexpr Kind kinds[2][3] = {{{64, 4, 4, 3.908f, 1.49f, 1.334f, 0.96f, 2.395f, 2.207f, 0.154f, 0.098f},
                                 {32, 4, 4, 3.865f, 0.812f, 0.548f, 0, 0.604f, 2.135f, 0.118f, 0},
                                 {32, 8, 8, 3.711f, 0.843f, 0.96f, 0, 0.898f, 1.991f, 0.138f, 0.065f}},
                                {{64, 4, 1, 3.255f, 0.434f, 0.166f, 0, 1.09f, 2.431f, 0.167f, 0.064f},
                                 {64, 8, 2, 3.183f, 0.581f, 0.404f, 0, 1.605f, 2.497f, 0.129f, 0.063f}}};
  const bool plain = epilogue == kGemmPlain, half = elem_size == 2;
  if ((int64_t)(N + R) * K > (int64_t)1 << 26) return {0, 0, 0, 0};
  const int step = half ? kStep16 : 32;
  GradsPlan best = {0, 0, 0, 0};
  const Plan pw = plan(N, K, R, true, elem_size), px = plan(R, K, N, plain || amax, elem_size);
  if (half && std::max(pw.tile, px.tile) > 64) return best;   // (larger tiles read less)
  float best_cost = (half ? 0.96f : 0.88f) * (pw.cost + px.cost);
  for (const Kind& kind : kinds[half]) {
    if (kind.tile == 0) break;
    const int tk = (K + kind.tile - 1) / kind.tile, tw = (N + kind.tile - 1) / kind.tile * tk, tx = (R + kind.tile - 1) / kind.tile * tk;
    if (amax && tx > kAmaxBlocks) continue;
    const float read = kind.read * 2e-6f * elem_size * kind.tile * ((float)tw * R + (float)tx * N), r2 = read * read;
    for (const int w : {1, 2, 3, 4, 6, 8, 12, 16}) {
      if (w > 1 && (w * 64 > R || tw * w > 1100)) break;
      const int nw = ((R + w - 1) / w + step - 1) / step;
      for (const int x : {1, 2, 4, 8}) {
        if (x > 1 && (!plain || amax || x * 128 > N || tx * x > 600)) break;
        if (kind.tile == 32 && tw * w + tx * x > 1280) continue;   // (all tiles of 32 x 32 read twice what those of 64 x 64 do)
        const int nx = ((N + x - 1) / x + step - 1) / step, tw_ = (nw + kind.turns - 1) / kind.turns, tx_ = (nx + kind.turns - 1) / kind.turns, longest = std::max(tw_, tx_);
        const float groups_w = (tw + 7) / 8 * w * (1 / 32.f), groups_x = (tx + 7) / 8 * x * (1 / 32.f);
        const float alone = kind.alone * longest + kind.end, all = kind.shared * std::max(groups_w * tw_ + groups_x * tx_, (float)longest) + kind.ends * std::ceil(groups_w + groups_x);
        const float a2 = alone * alone, s2 = all * all;
        const float cost = kind.start + std::sqrt(std::sqrt(a2 * a2 + s2 * s2 + r2 * r2)) + kind.split * ((w > 1) + (x > 1)) +
                           kind.split_mb * 8e-6f * ((w > 1 ? (float)w * N * K : 0) + (x > 1 ? (float)x * R * K : 0));
        if (cost < best_cost) { best_cost = cost; best = {kind.tile, kind.waves, w, x}; }
      }
    }
  }
  return best;
}
int64_t grads_workspace(int R, int N, int K, int elem_size, int epilogue, bool amax) {
  const GradsPlan g = grads_plan(R, N, K, elem_size, epilogue, amax);
  if (g.tile == 0) return -1;
  return ((g.w_splits > 1 ? (int64_t)g.w_splits * N * K : 0) + (g.x_splits > 1 ? (int64_t)g.x_splits * R * K : 0)) * 4;
}
int launch_grads(GradsArgs p, int dtype, float* workspace, PartSum* later, hipStream_t stream) {
  const int step = dtype == 0 ? 32 : kStep16;
  const GradsPlan g = grads_plan(p.x.M, p.x.K, p.x.N, dtype == 0 ? 4 : 2, p.x.epilogue, p.x.amax != nullptr);
  auto place = [&](GemmArgs& a, int splits, int& groups, int& row) {
    a.k_per_split = ((a.K + splits - 1) / splits + step - 1) / step * step;
    splits = (a.K + a.k_per_split - 1) / a.k_per_split;   // rounding up may leave the last ones empty
    a.part = splits > 1 ? workspace : nullptr;
    if (splits > 1) workspace += (int64_t)splits * a.M * a.N;
    row = (((a.M + g.tile - 1) / g.tile) * ((a.N + g.tile - 1) / g.tile) + 7) / 8 * 8;
    groups = row * splits;
  };
  place(p.w, g.w_splits, p.w_groups, p.w_row);
  place(p.x, g.x_splits, p.x_groups, p.x_row);
  int rc = dtype == 0 ? launch_grads32(p, g.tile, g.waves, stream) : by_type16(dtype, true, [&](auto t, auto) {
    using T = decltype(t);
    if (g.waves == 8) hipLaunchKernelGGL((grads_kernel<T, 2>), dim3(p.w_groups + p.x_groups), dim3(2 * kThreads), 0, stream, p);
    else hipLaunchKernelGGL((grads_kernel<T, 1>), dim3(p.w_groups + p.x_groups), dim3(kThreads), 0, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : -3;
  });
  PartSum sums[2];
  int count = 0;
  if (later != nullptr) later->parts = 0;
  for (const GemmArgs* a : {&p.w, &p.x}) {
    if (a->part == nullptr) continue;
    const PartSum sum = {a->part, (int64_t)a->M * a->N, a->c, (a->K + a->k_per_split - 1) / a->k_per_split, 0};
    if (a == &p.w && later != nullptr) *later = sum;
    else sums[count++] = sum;
  }
  if (rc == 0 && count > 0) rc = launch_sums(sums, count, dtype, stream);
  return rc;
}

}  // namespace castle
