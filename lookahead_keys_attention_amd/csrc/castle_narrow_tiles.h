// What the forward and the backward kernels over 32-row work items share (castle_narrow.hip, castle_narrow_bwd.hip).
#pragma once
#include "castle_tiles.h"
#include "castle_params.h"
#include "castle_profile.h"
#include "castle_tqv.h"
#include "castle_waves.h"
#include "castle_dispatch.h"
#include "castle_narrow.h"


namespace castle {

extern __shared__ __attribute__((aligned(16))) unsigned char castle_smem[];

// Two-phase copy of a 32 x COLS tile whose rows are contiguous in memory into a row-major LDS tile, by one wave: every
// load covers 1 KB of consecutive addresses.  (MFMA fragments straight from global memory touch 32 lines per
// load; a CU works through those one after the other, which made it the bottleneck of these kernels: the key kernel at
// 3 x 4 heads of 1000 rows took 68 us that way.)
// SCALAR: see load_at
template <typename T, int COLS, bool SCALAR = true> struct Flat32 {
  static constexpr int V = elem_traits<T>::vec16, VPR = COLS / V, N = 32 * VPR / 64, LD = lds_ld_tr<T>(COLS);
  vec<T, V> r[N];
  __device__ __forceinline__ void load(const T* rows) {
    if constexpr (SCALAR) {
      const global_bytes base = scalar_base(rows);
      const uint32_t at = lane_offset(lane_id() * 16);
#pragma unroll
      for (int n = 0; n < N; ++n) r[n] = *(const __attribute__((address_space(1))) vec<T, V>*)(base + at + 1024 * n);
    } else {
#pragma unroll
      for (int n = 0; n < N; ++n) r[n] = *reinterpret_cast<const vec<T, V>*>(rows + (lane_id() + 64 * n) * V);
    }
  }
  __device__ __forceinline__ void store(T* tile, float mul) const {
    const int lane = lane_id();
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int v = lane + 64 * n;
      vec<float, V> f = __builtin_convertvector(r[n], vec<float, V>);
#pragma unroll
      for (int e = 0; e < V; ++e) f[e] *= mul;
      *reinterpret_cast<vec<T, V>*>(tile + (v / VPR) * LD + (v % VPR) * V) = __builtin_convertvector(f, vec<T, V>);
    }
  }
  __device__ __forceinline__ void store(T* tile) const {
    const int lane = lane_id();
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int v = lane + 64 * n;
      *reinterpret_cast<vec<T, V>*>(tile + (v / VPR) * LD + (v % VPR) * V) = r[n];
    }
  }
};
// the natural fragments (row c on the lanes) of a snapshot tile (512 consecutive bytes per half wave), and their
// row-major copy in an LDS tile
template <typename T, int HD> __device__ __forceinline__ void load_snap32(frag<T> (&f)[HD / 16], const T* tile, int c, int g) {
#pragma unroll
  for (int s = 0; s < HD / 16; ++s) f[s] = ldg_snap_nat<T>(tile, c, 16 * s + 8 * g);
}
template <typename T, int HD> __device__ __forceinline__ void put_rows32(T* tile, const frag<T> (&f)[HD / 16], int c, int g) {
  constexpr int LD = lds_ld_tr<T>(HD);
#pragma unroll
  for (int s = 0; s < HD / 16; ++s) *reinterpret_cast<frag_mem<T>*>(tile + c * LD + 16 * s + 8 * g) = f[s];
}

template <typename T, int HD> constexpr int wave_tile_bytes() { return (int)sizeof(T) * 32 * lds_ld_tr<T>(HD); }
template <typename T> constexpr int kLdT64 = lds_ld_tr<T>(kNB);              // of a tile of T' rows
template <typename T> constexpr int t_tile_bytes() { return (int)sizeof(T) * 32 * kLdT64<T>; }
template <typename T> constexpr int kLdX = 32 + 16 / (int)sizeof(T);   // leading dimension of a 32-column LDS tile
// two waves per SIMD where the fragments of 16-bit operands leave room for it
template <typename T, int HD> constexpr int narrow_waves() { return sizeof(T) == 2 && HD <= 64 ? 2 : 1; }
template <typename T, int HD> __device__ __forceinline__ void narrow_item(int BH, int n, int cus, int& rank, int& bh) {
  if constexpr (narrow_waves<T, HD>() == 2) work_item_snake(BH, n, cus, rank, bh);
  else work_item(BH, rank, bh);
}

template <typename K> static bool raise_lds(K kernel, int bytes) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
}
// Eight waves on an item instead of four while that leaves no CU a second workgroup to run (16-bit, d <= 64: two waves fit a
// SIMD) and the walk is long enough to share: 1 head x 8000 rows, us with 4 / 8: scan 79 / 63, attn 105 / 84, key 294 / 224;
// 4 x 2500: 31 / 27, 40 / 34, 102 / 81.  Level at 10 tiles, slower at 4.  (The query kernel gains nothing: 169 / 166, 67 / 75.)
template <typename T, int HD> bool eight_waves(const CoreShape& s) {
  const int64_t tiles = (s.L + 31) / 32;
  return sizeof(T) == 2 && HD <= 64 && tiles >= 16 && tiles * s.B * s.H <= kNarrowCus * 5 / 4;
}

}  // namespace castle
