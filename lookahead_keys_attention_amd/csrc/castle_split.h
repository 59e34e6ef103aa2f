// fp32 operands on 16-bit matrix instructions: every operand is the sum of two fp16 numbers.
//
// The fp32 matrix instruction does 4096 flop in 64 cycles, the fp16 one 32768 in 32.  x = h + l with h = fp16(x), l = fp16(x - h)
// keeps 22 to 24 bits of x while l is a normal fp16 number, that is from |x| = 2^-2 up to 2^16; a product is then
// ah bh + ah bl + al bh (al bl is below 2^-22 of it) in three instructions with fp32 accumulation: 96 cycles instead of 512 for a 32 x 32
// tile and 16 of its contraction.  So operands are brought near the top of that range by powers of two first, which are exact and are
// taken out of the fp32 sums again:
//   operands of the call   by the largest finite |x| of 32 rows of the operand in a head, when the copies of the operands are made: a copy holds
//                          the halves, and what these are to be multiplied with.  An element below 2^-17 of that maximum keeps an absolute error
//                          of 2^-40 of the maximum instead of 2^-24 of itself.
//   U, G                   by the largest value of a snapshot tile (32 keys)
//   T'                     by the largest value of its block
//   dS, dSu, dZ            by the largest value of the tile of 32 x 32, found in registers
//   gates, weights         are at most 1: times 2^12
// Sums over tiles of different scales are formed per tile and added in fp32.
#pragma once
#include "castle_tiles.h"
#include "castle_params.h"

namespace castle {

struct split8 { frag<fp16_t> h, l; };   // an operand fragment

__device__ __forceinline__ split8 split(const vec<float, 8>& x) {
  split8 f;
  f.h = __builtin_convertvector(x, frag<fp16_t>);
  vec<float, 8> r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = __builtin_fmaf((float)f.h[e], -1.f, x[e]);   // exact
  f.l = __builtin_convertvector(r, frag<fp16_t>);
  return f;
}
__device__ __forceinline__ split8 zero_split() { return split8{zero_frag<fp16_t>(), zero_frag<fp16_t>()}; }
__device__ __forceinline__ void mma(acc_t& c, const split8& a, const split8& b) {
  mma(c, a.l, b.h);
  mma(c, a.h, b.l);
  mma(c, a.h, b.h);
}
// with the product of the low halves too: for the output, whose first rows are sums of few values (error at 33 rows 0.97 -> 0.91e-7)
__device__ __forceinline__ void mma_full(acc_t& c, const split8& a, const split8& b) {
  mma(c, a.l, b.l);
  mma(c, a, b);
}
// registers 8 s .. 8 s + 7 of an accumulator tile, times `mul`, as an operand (chained order)
__device__ __forceinline__ split8 chain_split(const acc_t& c, int s, float mul) {
  vec<float, 8> v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = c[8 * s + e] * mul;
  return split(v);
}
__device__ __forceinline__ split8 chain_split(const acc_t& c, int s) {   // of values that are in range
  vec<float, 8> v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = c[8 * s + e];
  return split(v);
}
// sum += mul * t
__device__ __forceinline__ void add_scaled(acc_t& sum, const acc_t& t, float mul) {
#pragma unroll
  for (int r = 0; r < 16; ++r) sum[r] = __builtin_fmaf(t[r], mul, sum[r]);
}

// ---- tiles in LDS: 32 rows of the high halves, then 32 rows of the low halves -----------------------------------------------------
template <int COLS> constexpr int split_ld() { return COLS + 8; }
template <int COLS> constexpr int split_plane() { return 32 * split_ld<COLS>(); }
template <int COLS> constexpr int split_tile_bytes() { return 2 * 2 * split_plane<COLS>(); }
// row `row`, columns col .. col + 7
template <int COLS> __device__ __forceinline__ split8 ld_nat_split(const fp16_t* tile, int row, int col) {
  constexpr int LD = split_ld<COLS>();
  return split8{ld_nat<fp16_t>(tile, LD, row, col), ld_nat<fp16_t>(tile + split_plane<COLS>(), LD, row, col)};
}
// column n0 + c, the 16 rows from contr0 in chained order (see ld_free)
template <int COLS> __device__ __forceinline__ split8 ld_free_split(const fp16_t* tile, int n0, int contr0, int c, int g) {
  constexpr int LD = split_ld<COLS>();
  return split8{ld_free<fp16_t, true>(tile, LD, n0, COLS, contr0, c, g), ld_free<fp16_t, true>(tile + split_plane<COLS>(), LD, n0, COLS, contr0, c, g)};
}

// ---- tiles in memory: the high halves of 32 rows, then the low ones, each in the order of the fragments: 16 columns after 16, lane after lane.  A
// fragment of rows is one load of 1 KB of consecutive addresses (the layout of the snapshot tiles). ---------------------------------------------
template <int COLS> constexpr int split_elems() { return 2 * 32 * COLS; }
template <int COLS> struct SplitRows {
  static constexpr int S = COLS / 16;
  split8 f[S];
  __device__ __forceinline__ void load(const fp16_t* tile) {
    const global_bytes base = scalar_base(tile);
    const uint32_t at = lane_offset(lane_id() * 16);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      f[s].h = *(const __attribute__((address_space(1))) frag<fp16_t>*)(base + at + 1024 * s);
      f[s].l = *(const __attribute__((address_space(1))) frag<fp16_t>*)(base + at + 1024 * (S + s));
    }
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int s = 0; s < S; ++s) f[s] = zero_split();
  }
  // into a padded LDS tile
  __device__ __forceinline__ void store(fp16_t* tile) const {
    const int c = lane_id() & 31, g = lane_id() >> 5;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      fp16_t* p = tile + c * split_ld<COLS>() + 16 * s + 8 * g;
      *reinterpret_cast<frag_mem<fp16_t>*>(p) = f[s].h;
      *reinterpret_cast<frag_mem<fp16_t>*>(p + split_plane<COLS>()) = f[s].l;
    }
  }
  // into LDS as it is, to be read with of_rows()
  __device__ __forceinline__ void store_flat(fp16_t* tile) const {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      *reinterpret_cast<frag_mem<fp16_t>*>(tile + 512 * s + 8 * lane_id()) = f[s].h;
      *reinterpret_cast<frag_mem<fp16_t>*>(tile + 512 * (S + s) + 8 * lane_id()) = f[s].l;
    }
  }
};
template <int COLS> __device__ __forceinline__ split8 of_rows(const fp16_t* flat, int s) {
  return split8{*reinterpret_cast<const frag_mem<fp16_t>*>(flat + 512 * s + 8 * lane_id()), *reinterpret_cast<const frag_mem<fp16_t>*>(flat + 512 * (COLS / 16 + s) + 8 * lane_id())};
}
// natural -> chained contraction order: columns 4 .. 7 of the lower lanes change places with columns 0 .. 3 of the upper ones
__device__ __forceinline__ frag<fp16_t> chained(const frag<fp16_t>& f) {
  typedef vec<uint32_t, 4> u4;
  u4 x = __builtin_bit_cast(u4, f);
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const auto y = __builtin_amdgcn_permlane32_swap(x[e], x[2 + e], false, false);
    x[e] = y[0];
    x[2 + e] = y[1];
  }
  return __builtin_bit_cast(frag<fp16_t>, x);
}
__device__ __forceinline__ split8 chained(const split8& f) { return split8{chained(f.h), chained(f.l)}; }

// ---- scales --------------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ float abs_max(const acc_t& x, float m = 0.f) {
#pragma unroll
  for (int r = 0; r < 16; ++r) m = fmaxf(m, fabsf(x[r]));
  return m;
}
// the largest m >= 0 of a wave: its bits
__device__ __forceinline__ uint32_t wave_max_bits(float m) {
#define CASTLE_ROR_(N_) m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m), 0x120 + N_, 0xf, 0xf, false)))
  CASTLE_ROR_(8);
  CASTLE_ROR_(4);
  CASTLE_ROR_(2);
  CASTLE_ROR_(1);
#undef CASTLE_ROR_
  const int b = __builtin_bit_cast(int, m);
  const uint32_t x0 = __builtin_amdgcn_readlane(b, 0), x1 = __builtin_amdgcn_readlane(b, 16), x2 = __builtin_amdgcn_readlane(b, 32), x3 = __builtin_amdgcn_readlane(b, 48);
  const uint32_t a = x0 > x1 ? x0 : x1, d = x2 > x3 ? x2 : x3;   // (numbers >= 0 are ordered like their bits)
  return a > d ? a : d;
}
// The power of two that places a maximum with these bits in [2^13, 2^14), and its inverse, which the halves are to be multiplied with
struct TileScale { float mul, inv; };
__device__ __forceinline__ TileScale tile_scale(uint32_t bits) {
  uint32_t e = bits & 0x7f800000u;
  e = e < (31u << 23) ? 31u << 23 : e;
  return TileScale{__builtin_bit_cast(float, (267u << 23) - e), __builtin_bit_cast(float, e - (13u << 23))};
}
constexpr float kUnit = 4096.f, kUnitInv = 1.f / 4096.f;   // scale of gates and weights

// A tile of 32 fp32 rows, eight columns of a row per piece (piece lane + 64 n of the tile, row by row), into memory; returns what its halves are to be
// multiplied with
template <int COLS> __device__ __forceinline__ float store_split_tile(fp16_t* tile, const vec<float, 8> (&x)[COLS / 16]) {
  float m = 0.f;
#pragma unroll
  for (int n = 0; n < COLS / 16; ++n)
#pragma unroll
    for (int e = 0; e < 8; ++e) m = fmaxf(m, fabsf(x[n][e]));
  uint32_t bits = wave_max_bits(m);
  if (bits >= 0x7f800000u) {   // the largest finite one
    m = 0.f;
#pragma unroll
    for (int n = 0; n < COLS / 16; ++n)
#pragma unroll
      for (int e = 0; e < 8; ++e) m = fabsf(x[n][e]) <= __FLT_MAX__ ? fmaxf(m, fabsf(x[n][e])) : m;
    bits = wave_max_bits(m);
  }
  const TileScale s = tile_scale(bits);
#pragma unroll
  for (int n = 0; n < COLS / 16; ++n) {
    const int q = lane_id() + 64 * n;
    const split8 f = split(x[n] * s.mul);
    fp16_t* p = tile + snap_elem<fp16_t>(q / (COLS / 8), q % (COLS / 8) * 8);
    *reinterpret_cast<frag_mem<fp16_t>*>(p) = f.h;
    *reinterpret_cast<frag_mem<fp16_t>*>(p + 32 * COLS) = f.l;
  }
  return s.inv;
}
// the operands of a call, in this order, and a head's tiles of one of them
enum { kOpQc, kOpKc, kOpVc, kOpQu, kOpKu, kOpVu };
template <int HD> __device__ __forceinline__ const fp16_t* split_tiles(const void* copy, int bh, int tiles) {
  return reinterpret_cast<const fp16_t*>(copy) + (int64_t)bh * tiles * split_elems<HD>();
}
template <int HD> __device__ __forceinline__ fp16_t* split_tiles_mut(void* copy, int bh, int tiles) {
  return reinterpret_cast<fp16_t*>(copy) + (int64_t)bh * tiles * split_elems<HD>();
}

}  // namespace castle
