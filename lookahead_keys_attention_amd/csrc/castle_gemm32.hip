// Products of fp32 operands on the 16-bit matrix instructions.
//
// An element is three bf16 numbers, x = a + b + c exactly (8 of its 24 bits in each, any exponent), and a product is
//   ac' + ca' + bb' + ab' + ba' + aa'
// with fp32 sums: 192 cycles for a tile of 32 x 32 and 16 steps of the contraction, where the fp32 instruction takes 512 and rounds its sums four times as
// often.  What is left out, bc' + cb' + cc', is below 2^-23 of a product, of either sign.  Infinities, NaNs and what bf16 rounds to infinity do not go by parts; they
// leave no finite sum, and a wave that finds such a one goes over its steps again with the fp32 instruction.  So it does where a sum is below 2^-90 and not zero: of an
// element below 2^-110, c is below what bf16 holds, 2^-133, an error of up to 2^-134.  In a sum of 2^-90 or more that is below 2^-24 of it, as long as the other operand's
// elements add up to no more than 2^20.
//
// A workgroup has a tile of 64 x 64 or 32 x 32 of the output, and its waves take the contraction in turns, 32 steps each: every wave meets the whole tile, so an
// element is converted once for it, six matrix instructions follow on two to four operands, and the operands go through LDS that belongs to the wave, with no barrier
// before the sums of the waves are added.  (The tile in quarters, one to a wave, with the parts in LDS was slower than the fp32 instruction: conversion, LDS and matrix
// instructions took 480, 576 and 384 cycles a step of 32, one behind the other.  Operands straight from memory into registers: four times the requests, 680 cycles for 16 steps
// of a tile of 64 against 470.)
// What bounds a large product is conversion and matrix instructions together, 1400 and 1540 cycles for a wave's 32 steps of a tile of 64: of two waves on a SIMD
// one's vector instructions hide only two thirds of their time behind the other's matrix instructions; a small one, its start, one trip to memory and the sums.
// us, on the fp32 instruction / here, by rows: 256 rows 512 -> 3072 forward 14.0 / 12.7, input gradient 16.1 / 14.7, weight gradient 15.9 / 11.4, 512 -> 512 8.4 / 5.6, 8.7 / 5.8,
// 9.1 / 4.9; 16384 rows 512 -> 3072 441 / 303, 431 / 323, 506 / 302.  2-norm error against 64 bits, units of 1e-7, the same way: 512 -> 3072 2.9 / 1.7 to 4.1 / 3.4 forward,
// weight gradient of 20 rows 0.82 / 0.65, of 16384 16 / 7.6.
#include "castle_tiles.h"
#include "castle_gemm.h"
#include "castle_gelu.h"
#include "castle_waves.h"
#include <type_traits>

namespace castle {
namespace {

struct split3 { frag<bf16_t> a, b, c; };
typedef vec<float, 8> raw8;
__device__ __forceinline__ split3 split_in_three(raw8 x) {
  typedef vec<uint32_t, 4> words;
  // `f` of pairs leaves x, exactly
  auto part = [&](auto&& f, bool rest) __attribute__((always_inline)) {
    words p;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t w = f(x[2 * e], x[2 * e + 1]);
      p[e] = w;
      if (rest) {
        x[2 * e] -= __builtin_bit_cast(float, w << 16);
        x[2 * e + 1] -= __builtin_bit_cast(float, w & 0xffff0000);
      }
    }
    return __builtin_bit_cast(frag<bf16_t>, p);
  };
  auto rounded = [](float lo, float hi) __attribute__((always_inline)) {
    uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(vec<float, 2>{lo, hi}, vec<bf16_t, 2>));
    asm("" : "+v"(w));   // or each is rounded by itself, and once more in the pair
    return w;
  };
  // upper halves: the conversion takes as long as two other instructions
  auto cut = [](float lo, float hi) __attribute__((always_inline)) { return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, hi), __builtin_bit_cast(uint32_t, lo), 0x07060302); };
  split3 s;
  s.a = part(rounded, true);
  s.b = part(cut, true);
  s.c = part(cut, false);
  return s;
}

// 32 or 64 rows or columns of an operand and 32 steps of the contraction, 4 or 8 KB: straight from memory to LDS in pieces of 16 bytes, then as fragments of raw elements to
// the registers of the same wave.  KC: contraction-contiguous, else [contraction][free].  Rows cannot be padded, since pieces go to LDS in the order of the lanes:
// they take other places in their rows, such that the lanes of a read meet all banks (KC: piece p of row r at p ^ (r / 2 % 8); else the halves of row k swapped
// where k / 8 is odd, or of 32 the rows k and k ^ 1).  Pieces beyond the free end read another row's data: those outputs are not stored.
constexpr int kStep = 32;
template <bool KC, int F> struct Operand32 {   // F: 32 or 64
  static constexpr int kBytes = F * kStep * 4, kLoads = kBytes / 1024, PIECES = F / 4;
  const float* base;
  int last;   // row or column of the tile that is still there
  uint32_t at[kLoads];
  static __device__ __forceinline__ int turn(int k) { return F == 64 ? 8 * (k >> 3 & 1) : 0; }   // pieces
  static __device__ __forceinline__ int row_of(int k) { return F == 32 ? k ^ (k >> 3 & 1) : k; }
  __device__ __forceinline__ uint32_t place(int ld, int q, int steps) const {   // of the piece that this lane fetches; steps: what is left of the contraction
    const int lane = lane_id();
    if constexpr (KC) {
      const int row = 8 * q + (lane >> 3), piece = (lane & 7) ^ (row >> 1 & 7);
      return 4 * (uint32_t)(min(row, last) * ld + (4 * piece < steps ? 4 * piece : 0));
    } else {
      const int k = row_of(64 / PIECES * q + lane / PIECES), piece = lane % PIECES ^ turn(k);
      return 4 * (uint32_t)(min(k, steps - 1) * ld + (4 * piece <= last ? 4 * piece : 0));
    }
  }
  __device__ __forceinline__ void start(const float* p, int64_t ld, int free0, int free_end) {
    base = p + (KC ? free0 * ld : free0);
    last = free_end - 1 - free0;
#pragma unroll
    for (int q = 0; q < kLoads; ++q) at[q] = place((int)ld, q, kStep);
  }
  __device__ __forceinline__ void load(int64_t ld, int k, int k_end, uint32_t lds) const {
    const float* p = base + (KC ? k : k * ld);
    if (k + kStep <= k_end) {
#pragma unroll
      for (int q = 0; q < kLoads; ++q) load_to_lds(p, at[q], lds + 1024 * q);
    } else {
#pragma unroll
      for (int q = 0; q < kLoads; ++q) load_to_lds(p, place((int)ld, q, k_end - k), lds + 1024 * q);
    }
  }
  // 16 steps from 16 s; steps: what is left of the contraction, zeros behind it
  static __device__ __forceinline__ void read(const float* lds, raw8 (&x)[F / 32], int s, int steps, int c, int g) {
    typedef vec<float, 4> v4;
#pragma unroll
    for (int i = 0; i < F / 32; ++i) {
      if constexpr (KC) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const v4 q = *reinterpret_cast<const v4*>(lds + (32 * i + c) * kStep + 4 * ((4 * s + 2 * g + h) ^ (c >> 1 & 7)));
#pragma unroll
          for (int e = 0; e < 4; ++e) x[i][4 * h + e] = q[e];
        }
      } else if constexpr (F == 64) {
        const float* p = lds + 8 * g * F + ((32 * i + c) ^ 32 * g);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[i][e] = p[(16 * s + e) * F];
      } else {
        const float* p[2] = {lds + (8 * g + g) * F + c, lds + (8 * g + 1 - g) * F + c};
#pragma unroll
        for (int e = 0; e < 8; ++e) x[i][e] = p[e & 1][(16 * s + (e & ~1)) * F];
      }
    }
    if (steps < kStep) {
#pragma unroll
      for (int i = 0; i < F / 32; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (16 * s + 8 * g + e >= steps) x[i][e] = 0.f;
    }
  }
};

// sums of a wave in LDS: pieces of 16 bytes from one quad of accumulator registers to the next, such that the readers' pieces of a row meet all banks
constexpr int kUnit32 = 66;
constexpr uint32_t kLeastBits = (127u - 90) << 23;   // 2^-90
template <int TILE> constexpr int wave_bytes() { return max2(TILE * TILE / 256 * kUnit32 * 16, 2 * TILE * kStep * 4); }
// NORM: the rows of `a` are normalised on their way to the registers.
template <bool AK, bool BKC, int TILE, int W, bool NORM>
__device__ __forceinline__ void gemm32_tile(const GemmArgs& a, vec<float, 4>* s_sum, int bx, int by) {   // s_sum: of a wave, operands, then sums
  constexpr int V = 4, NT = 64 * W, BM = TILE, BN = TILE, F = TILE / 32, U = 4 * F * F;   // U: quads of accumulator registers
  typedef Operand32<AK, TILE> OpA;
  typedef Operand32<BKC, TILE> OpB;
  typedef vec<float, 4> v4;
  constexpr int kWave = wave_bytes<TILE>() / 16;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  // XCD x takes the x-th eighth of the tiles, for its L2
  const int tiles_n = (a.N + BN - 1) / BN, tiles = (a.M + BM - 1) / BM * tiles_n, share = (tiles + 7) / 8;
  const int tile = bx % 8 * share + bx / 8;
  if (tile >= tiles) return;
  const int m0 = tile / tiles_n * BM, n0 = tile % tiles_n * BN;
  const int k0 = by * a.k_per_split, k_end = min(a.K, k0 + a.k_per_split), stages = (k_end - k0 + kStep - 1) / kStep;
  const int amax_tile = a.amax_from / BN, amax_tiles = (a.amax_to - 1) / BN + 1 - amax_tile;   // of a row of tiles
  if (a.amax != nullptr && bx == 0) {
    for (int i = (a.M + BM - 1) / BM * amax_tiles + threadIdx.x; i < kAmaxBlocks; i += NT) a.amax[i] = 0.f;
    if (threadIdx.x == 0 && a.amax_status != nullptr) *a.amax_status = 0;
  }
  OpA oa;
  OpB ob;
  oa.start(static_cast<const float*>(a.a), a.lda, m0, a.M);
  ob.start(static_cast<const float*>(a.b), a.ldb, n0, a.N);
  const float* const mine = reinterpret_cast<const float*>(s_sum + wave * kWave);
  const uint32_t lds = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) float*)mine;
  auto fetch = [&](int stage) __attribute__((always_inline)) {
    if (stage >= stages) return;
    oa.load(a.lda, k0 + kStep * stage, k_end, lds);
    ob.load(a.ldb, k0 + kStep * stage, k_end, lds + OpA::kBytes);
  };
  fetch(wave);
  __shared__ __attribute__((aligned(16))) float s_norm[NORM ? kNormBytes / 4 : 4], s_factor[NORM ? BM : 1];
  const bool norm_keeps = NORM && a.h != nullptr && n0 == 0;   // (the first column of tiles stores what all of them form)
  float factor[F];
  if constexpr (NORM) {
    constexpr int LPR = NT / BM < 16 ? NT / BM : 16;   // lanes of a row
    const int row = threadIdx.x / LPR, sub = threadIdx.x % LPR;
    const float* x = static_cast<const float*>(a.a) + (int64_t)min(m0 + row, a.M - 1) * a.lda;
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
          const v4 f = *reinterpret_cast<const v4*>(x + (i < pieces ? i : 0) * V);
#pragma unroll
          for (int e = 0; e < V; ++e) {
            const float y = i < pieces ? f[e] : 0.f;
            sum[v] = __builtin_fmaf(y, y, sum[v]);
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
    for (int i = threadIdx.x; i < a.K; i += NT) s_norm[i] = static_cast<const float*>(a.norm_w)[i];
#pragma unroll
    for (int o = 1; o < LPR; o <<= 1) ssq += __shfl_xor(ssq, o);
    const float r = 1.f / sqrtf(ssq / (float)a.K + a.eps);
    if (sub == 0) {
      s_factor[row] = r;
      if (norm_keeps && a.rstd != nullptr && m0 + row < a.M) a.rstd[m0 + row] = r;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < F; ++i) factor[i] = s_factor[32 * i + c];
  }
  acc_t acc[F][F];   // [n rows, m lanes]
  auto products = [&](auto by_parts) __attribute__((always_inline)) {
    constexpr bool PARTS = decltype(by_parts)::value;
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int j = 0; j < F; ++j) zero(acc[i][j]);
    for (int stage = wave; stage < stages; stage += W) {
      const int k = k0 + kStep * stage;
      raw8 xa[2][F], xb[2][F];
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        OpA::read(mine, xa[s], s, k_end - k, c, g);
        OpB::read(mine + OpA::kBytes / 4, xb[s], s, k_end - k, c, g);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      fetch(stage + W);
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        if constexpr (NORM) {
          const int col = k + 16 * s + 8 * g;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if (col + 4 * h >= k_end) continue;
            const v4 w = *reinterpret_cast<const v4*>(s_norm + col + 4 * h);
#pragma unroll
            for (int i = 0; i < F; ++i) {
              v4 y;
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                y[e] = xa[s][i][4 * h + e] * factor[i] * w[e];
                xa[s][i][4 * h + e] = y[e];
              }
              if (norm_keeps && m0 + 32 * i + c < a.M) *reinterpret_cast<v4*>(static_cast<float*>(a.h) + (int64_t)(m0 + 32 * i + c) * a.K + col + 4 * h) = y;
            }
          }
        }
        if constexpr (PARTS) {
          split3 fa[F], fb[F];
#pragma unroll
          for (int i = 0; i < F; ++i) {
            fa[i] = split_in_three(xa[s][i]);
            fb[i] = split_in_three(xb[s][i]);
          }
#pragma unroll
          for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j) {
              castle::mma(acc[i][j], fb[j].c, fa[i].a);
              castle::mma(acc[i][j], fb[j].a, fa[i].c);
              castle::mma(acc[i][j], fb[j].b, fa[i].b);
              castle::mma(acc[i][j], fb[j].b, fa[i].a);
              castle::mma(acc[i][j], fb[j].a, fa[i].b);
              castle::mma(acc[i][j], fb[j].a, fa[i].a);
            }
        } else {
#pragma unroll
          for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j) castle::mma(acc[i][j], __builtin_bit_cast(frag<float>, xb[s][j]), __builtin_bit_cast(frag<float>, xa[s][i]));
        }
      }
    }
    settle();
  };
  products(std::true_type());
  float most = 0.f;
  // the place of |sum| above kLeast; smaller ones are beyond infinity
  auto above = [&](bool zeros_count) __attribute__((always_inline)) {
    uint32_t far = 0;
#pragma unroll
    for (int i = 0; i < F * F; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float x = acc[i / F][i % F][r];   // (the bits of an element of a vector are taken from a copy: from the element itself they are the first one's)
        const uint32_t w = 2 * __builtin_bit_cast(uint32_t, x);
        far = max(far, (!zeros_count && w == 0 ? 2 * kLeastBits : w) - 2 * kLeastBits);
      }
    return far >= 2 * (0x7f800000u - kLeastBits);
  };
  // (zeros, of rows of zeros for instance, are looked at by themselves: that costs another instruction for each sum)
  if (__builtin_amdgcn_ballot_w64(above(true)) != 0 && __builtin_amdgcn_ballot_w64(above(false)) != 0) {
    fetch(wave);
    products(std::false_type());
  }
  // ---- sums of the waves that had a part of the contraction -------------------------------------------------------------------
  const int with = min(W, stages);
  __syncthreads();   // the operands are read
  if (wave < with) {
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int j = 0; j < F; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) s_sum[wave * kWave + (4 * (F * i + j) + q) * kUnit32 + 33 * g + c] = pack4<float>(acc[i][j], q);
  }
  __syncthreads();
#pragma unroll
  for (int u = threadIdx.x; u < BM * BN / 4; u += NT) {
    const int row = u / (BN / 4), p = u % (BN / 4), m = m0 + row, n = n0 + 4 * p;
    if (m >= a.M || n >= a.N) continue;
    const v4* part = s_sum + (row / 32 * (4 * F) + p / 2) * kUnit32 + 33 * (p % 2) + row % 32;
    v4 x = part[0];
    for (int w = 1; w < with; ++w) x += part[w * kWave];
    if (a.part != nullptr) {   // partial product of this range of the contraction
      *reinterpret_cast<v4*>(a.part + (int64_t)by * a.M * a.N + (int64_t)m * a.N + n) = x;
      continue;
    }
    const int64_t at = (int64_t)m * a.ldc + n;
    if (a.epilogue == kGemmGeluSlope) {
      const v4 y = *reinterpret_cast<const v4*>(static_cast<const float*>(a.aux) + at);
#pragma unroll
      for (int e = 0; e < V; ++e) x[e] *= gelu_slope<float>(y[e]);
    }
    *reinterpret_cast<v4*>(static_cast<float*>(a.c) + at) = x;
    if (a.amax != nullptr && n >= a.amax_from && n < a.amax_to) {
#pragma unroll
      for (int e = 0; e < V; ++e) most = fmaxf(most, fabsf(x[e]));   // fmaxf drops NaNs
    }
    if (a.epilogue == kGemmGelu) {
#pragma unroll
      for (int e = 0; e < V; ++e) x[e] = gelu<float>(x[e]);
      *reinterpret_cast<v4*>(static_cast<float*>(a.aux) + at) = x;
    }
  }
  const int slot = n0 / BN - amax_tile;
  if (a.amax != nullptr && slot >= 0 && slot < amax_tiles) {
    __shared__ float s_most[W];
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) most = fmaxf(most, __shfl_xor(most, o));
    if (lane == 0) s_most[wave] = most;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int w = 1; w < W; ++w) most = fmaxf(most, s_most[w]);
      a.amax[m0 / BM * amax_tiles + slot] = fminf(most, 3.0e38f);   // an infinite value counts as the largest finite one
    }
  }
}
template <bool AK, bool BKC, int TILE, int W, bool NORM>
__global__ __launch_bounds__(64 * W, W / 4 < 2 ? 2 : W / 4) void gemm32_kernel(GemmArgs a) {
  __shared__ __attribute__((aligned(16))) vec<float, 4> s_sum[W * wave_bytes<TILE>() / 16];
  gemm32_tile<AK, BKC, TILE, W, NORM>(a, s_sum, blockIdx.x, blockIdx.y);
}
// both gradients of a projection: workgroups of the weight gradient, then those of the input gradient (castle_gemm.hip; 256 rows 512 -> 3072, us: 12.9 and 16.1, both
// 24.6, 512 -> 512 5.6 and 6.5, both 8.4)
template <int TILE, int W> __global__ __launch_bounds__(64 * W, W / 4 < 2 ? 2 : W / 4) void grads32_kernel(GradsArgs p) {
  __shared__ __attribute__((aligned(16))) vec<float, 4> s_sum[W * wave_bytes<TILE>() / 16];
  int b = blockIdx.x;
  if (b < p.w_groups) {
    gemm32_tile<false, false, TILE, W, false>(p.w, s_sum, b % p.w_row, b / p.w_row);
  } else {
    b -= p.w_groups;
    gemm32_tile<true, false, TILE, W, false>(p.x, s_sum, b % p.x_row, b / p.x_row);
  }
}

}  // namespace

int launch_gemm32(const GemmArgs& a, bool a_kc, bool b_kc, int tile, int splits, int waves, hipStream_t stream) {
  const int tiles = ((a.M + tile - 1) / tile) * ((a.N + tile - 1) / tile);
  const dim3 grid((tiles + 7) / 8 * 8, splits);
  auto go = [&](auto ak, auto bk, auto norm) {
    constexpr bool AK = decltype(ak)::value, BKC = decltype(bk)::value, NORM = decltype(norm)::value;
    if (tile == 32 && waves == 8) hipLaunchKernelGGL((gemm32_kernel<AK, BKC, 32, 8, NORM>), grid, dim3(512), 0, stream, a);
    else if (tile == 32) hipLaunchKernelGGL((gemm32_kernel<AK, BKC, 32, 4, NORM>), grid, dim3(256), 0, stream, a);
    else if (waves == 4) hipLaunchKernelGGL((gemm32_kernel<AK, BKC, 64, 4, NORM>), grid, dim3(256), 0, stream, a);
    else if constexpr (NORM) return -2;
    else if (waves == 2) hipLaunchKernelGGL((gemm32_kernel<AK, BKC, 64, 2, NORM>), grid, dim3(128), 0, stream, a);
    else hipLaunchKernelGGL((gemm32_kernel<AK, BKC, 64, 1, NORM>), grid, dim3(64), 0, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -3;
  };
  const std::true_type yes{};
  const std::false_type no{};
  if (a.norm_w != nullptr) return go(yes, yes, yes);
  if (a_kc) return b_kc ? go(yes, yes, no) : go(yes, no, no);
  return b_kc ? -2 : go(no, no, no);
}

int launch_grads32(const GradsArgs& p, int tile, int waves, hipStream_t stream) {
  const dim3 grid(p.w_groups + p.x_groups);
  if (tile == 32 && waves == 8) hipLaunchKernelGGL((grads32_kernel<32, 8>), grid, dim3(512), 0, stream, p);
  else if (tile == 32) hipLaunchKernelGGL((grads32_kernel<32, 4>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((grads32_kernel<64, 4>), grid, dim3(256), 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

}  // namespace castle
