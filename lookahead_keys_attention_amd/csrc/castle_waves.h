// What the kernels over 32-row work items share: waits, order of LDS traffic inside a wave, sums over the waves of a workgroup,
// gradient stores.
#pragma once
#include "castle_tiles.h"

namespace castle {

// Waits out the longest matrix instruction (see the note on branches in castle_narrow.hip): in front of the first reads of accumulators
// whose last product sits in a loop or a branch that has just ended.
__device__ __forceinline__ void settle() {
  asm volatile("s_nop 15\n\ts_nop 3" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// the compiler waits for every load in flight at each read of LDS if it knows of loads into it: it is not told
__device__ __forceinline__ void load_to_lds(const void* base, uint32_t offset, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(offset), "s"(base) : "memory", "m0");
}
// LDS traffic of one wave is in order; this keeps the compiler from moving it (and, where registers are short, from
// requesting operands of the next stage early)
template <bool STAGES = false> __device__ __forceinline__ void wave_lds_order() {
  asm volatile("" ::: "memory");
  if constexpr (STAGES) __builtin_amdgcn_sched_barrier(0);
}

// Sums accumulator tiles over the W waves of a workgroup; wave w hands the quads q % W == w (four consecutive rows
// n = 32 nt + 8 q + 4 g .. of the lane's column) to f(nt, q, sum)
template <int W, int NT, typename F>
__device__ __forceinline__ void reduce_waves(float* lds, const acc_t (&acc)[NT], int wave, int lane, F&& f) {
  typedef vec<float, 4> v4;
  v4* s = reinterpret_cast<v4*>(lds);
  settle();
  __syncthreads();   // whatever the memory held before is dead
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int q = 0; q < 4; ++q) s[(wave * NT * 4 + nt * 4 + q) * 64 + lane] = v4{acc[nt][4 * q], acc[nt][4 * q + 1], acc[nt][4 * q + 2], acc[nt][4 * q + 3]};
  __syncthreads();
#pragma unroll
  for (int t = 0; t < NT * 4; ++t) {
    if (t % W != wave) continue;
    v4 sum = s[t * 64 + lane];
#pragma unroll
    for (int w = 1; w < W; ++w) sum += s[(w * NT * 4 + t) * 64 + lane];
    f(t / 4, t % 4, sum);
  }
}

// the sum of one accumulator tile over the waves, in every wave
template <int W> __device__ __forceinline__ void total_of_waves(float* lds, acc_t& acc, int wave, int lane) {
  typedef vec<float, 4> v4;
  v4* s = reinterpret_cast<v4*>(lds);
  settle();
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) s[(wave * 4 + q) * 64 + lane] = v4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    v4 sum = s[q * 64 + lane];
#pragma unroll
    for (int w = 1; w < W; ++w) sum += s[(w * 4 + q) * 64 + lane];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[4 * q + e] = sum[e];
  }
}

// four consecutive columns n .. n + 3 of a gradient row, rotated back (pos >= 0) and scaled
template <typename TI, int HD> __device__ __forceinline__ void store_quad(TI* row, int n, vec<float, 4> v, float mul, int pos) {
  if (n >= HD) return;
  if (pos >= 0) {
    CASTLE_ROPE_PAIR(v[0], v[1], (float)pos, n / 2, HD, true);
    CASTLE_ROPE_PAIR(v[2], v[3], (float)pos, n / 2 + 1, HD, true);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] *= mul;
  st4<TI>(row + n, __builtin_convertvector(v, vec<TI, 4>));
}

template <int HD> constexpr int narrow_nt() { return (HD < 32 ? 32 : HD) / 32; }
template <int HD, int W> constexpr int reduce_bytes() { return W * narrow_nt<HD>() * 16 * 64 * 4; }
constexpr int max2(int a, int b) { return a > b ? a : b; }

}  // namespace castle
