// The forward pass of short sequences, of which no backward pass follows, in one launch: a workgroup per 32 queries of a head.
//
// Up to 128 rows the four launches of the general path (operand copies, states and T' blocks, attention) cost 3 to 6 us each and are over before they
// have filled the GPU.  Here the rows that a query tile meets lie in LDS (converted, scaled and rotated on the way) and nothing goes through memory in
// between; there are no states to carry either: a key tile meets all sources between itself and the queries at once,
//   Su'[i, k] = sum over source tiles jt of  A[k, jt] T'[i, jt]^T.
// Wave w takes key tile w % 4 and every second source tile; the two halves of Su' are added through LDS, the key tiles merged at the end.  Every
// workgroup converts its rows by itself: what bounds the launch is latency (arguments, one trip to memory, conversion, two gates, a score tile,
// the merge), and that all heads and tiles run side by side.  Device time of the pass, us, general path / this one, bf16, d = 64, by heads x rows:
// 8 x 32 16.2 / 8.6, 8 x 128 17.2 / 10.7, 128 x 64 24.4 / 9.5, 256 x 96 33.9 / 28.0, 4096 x 64 389 / 119; d = 128, 8 x 96 22.2 / 13.0.
// A layer's forward (hidden 512, 8 heads, 64 tokens, with both projections) 25.8 / 19.9, which is the host's time for it.
#include "castle_tiles.h"
#include "castle_params.h"
#include "castle_profile.h"
#include "castle_dispatch.h"
#include "castle_waves.h"
#include "castle_narrow.h"

namespace castle {

extern __shared__ __attribute__((aligned(16))) unsigned char castle_smem[];

constexpr int kShortTiles = 4, kShortThreads = 512;   // two waves to a tile of 32 keys
// five operands of all rows, one tile of queries and half of the score sums; the merge reuses the whole of it
template <typename T, int HD> constexpr int short_lds(int tiles) {
  return max2((5 * tiles + 1) * 32 * lds_ld<T>(HD) * (int)sizeof(T) + kShortTiles * 64 * 16 * 4, kShortTiles * 64 * (narrow_nt<HD>() * 16 + 2) * 4);
}
// the largest m of a wave
__device__ __forceinline__ float wave_max(float m) {
#define CASTLE_ROR_(N_) m = fmaxf(m, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, m), 0x120 + N_, 0xf, 0xf, false)))
  CASTLE_ROR_(8);
  CASTLE_ROR_(4);
  CASTLE_ROR_(2);
  CASTLE_ROR_(1);
#undef CASTLE_ROR_
  const int b = __builtin_bit_cast(int, m);
  auto at = [&](int l) __attribute__((always_inline)) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(b, l)); };
  return fmaxf(fmaxf(at(0), at(16)), fmaxf(at(32), at(48)));
}

template <typename T, typename TI, int HD, bool ROTARY>
__global__ __launch_bounds__(kShortThreads, 2) void short_kernel(FwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>(), LD = lds_ld<T>(HD), V = elem_traits<T>::vec16, VPR = HD / V;
  constexpr bool CLAMP = __is_same(T, fp16_t) && !__is_same(TI, fp16_t);
  typedef vec<float, V> vf;
  const int L = a.s.L, tiles = (L + 31) / 32, it = tiles - 1 - (int)blockIdx.x % tiles, bh = blockIdx.x / tiles;
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const float c1 = a.s.scale * kLog2e;
  const bool want_u = a.U.ptr != nullptr;
  __shared__ float s_amax[kShortThreads / 64];
  T* const s_qc = reinterpret_cast<T*>(castle_smem);   // 32 rows; the others from row 0 on
  const int all = 32 * tiles * LD;
  T *const s_kc = s_qc + 32 * LD, *const s_vc = s_kc + all, *const s_qu = s_vc + all, *const s_ku = s_qu + all, *const s_vu = s_ku + all;
  float* const s_sum = reinterpret_cast<float*>(s_vu + all);
  // ---- operands ---------------------------------------------------------------------------------------------------------
  // rows up to the query tile's last; for the lookahead keys of the tile the sources behind it too
  const int seen = 32 * (it + 1), sources = want_u ? 32 * tiles : seen;
  constexpr int N = 32 * kShortTiles * VPR / kShortThreads > 0 ? 32 * kShortTiles * VPR / kShortThreads : 1;   // pieces of an operand per thread
  const View4 src[5] = {a.vu, a.ku, a.kc, a.qu, a.vc};
  const bool takes_q = threadIdx.x < 32 * VPR;   // (VPR is at most 16)
  vec<TI, V> x[5][N], xq;
#pragma unroll
  for (int e = 0; e < V; ++e) xq[e] = (TI)0.f;
#pragma unroll
  for (int o = 0; o < 5; ++o)
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int p = threadIdx.x + n * kShortThreads, row = p / VPR;
#pragma unroll
      for (int e = 0; e < V; ++e) x[o][n][e] = (TI)0.f;
      if (row < min(L, o < 2 ? sources : seen)) x[o][n] = *reinterpret_cast<const vec<TI, V>*>(head_ptr<TI>(src[o], b, h) + row * src[o].sl + p % VPR * V);
    }
  if (takes_q && 32 * it + (int)threadIdx.x / VPR < L)
    xq = *reinterpret_cast<const vec<TI, V>*>(head_ptr<TI>(a.qc, b, h) + (32 * it + threadIdx.x / VPR) * a.qc.sl + threadIdx.x % VPR * V);
  float most = 0.f;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const vf f = __builtin_convertvector(x[0][n], vf);
#pragma unroll
    for (int e = 0; e < V; ++e) most = fmaxf(most, fabsf(f[e]));   // drops NaNs
  }
  most = wave_max(most);
  if (lane == 0) s_amax[wave] = most;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < kShortThreads / 64; ++w) most = fmaxf(most, s_amax[w]);
  const float vu_scale = vu_scale_for(fminf(most, 3.0e38f), L), su_mul = 1.f / vu_scale;   // as in the general path, by workgroup
  float top = 0.f;   // of all that is stored: clamped, and reported, if it is beyond the fp16 range
  auto put = [&](T* to, const vec<TI, V>& raw, float mul, bool turn, int pos, int col) __attribute__((always_inline)) {
    vf f = __builtin_convertvector(raw, vf);
    if (ROTARY && turn) {
#pragma unroll
      for (int e = 0; e < V / 2; ++e) CASTLE_ROPE_PAIR(f[2 * e], f[2 * e + 1], (float)pos, col / 2 + e, HD, false);
    }
    float large = 0.f;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      f[e] *= mul;
      if constexpr (CLAMP) large = fmaxf(large, fabsf(f[e]));
    }
    if constexpr (CLAMP) {
      top = fmaxf(top, large);
      if (__builtin_amdgcn_ballot_w64(large > kHalfMax) != 0) {
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = __builtin_amdgcn_fmed3f(f[e], -kHalfMax, kHalfMax);
      }
    }
    *reinterpret_cast<vec<T, V>*>(to + col) = __builtin_convertvector(f, vec<T, V>);
  };
#pragma unroll
  for (int o = 0; o < 5; ++o) {
    T* const to = o == 0 ? s_vu : o == 1 ? s_ku : o == 2 ? s_kc : o == 3 ? s_qu : s_vc;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const int p = threadIdx.x + n * kShortThreads, row = p / VPR;
      if (row < (o < 2 ? sources : seen)) put(to + row * LD, x[o][n], o == 0 ? vu_scale : o == 1 ? -c1 : 1.f, o != 4, row, p % VPR * V);
    }
  }
  if (takes_q) put(s_qc + threadIdx.x / VPR * LD, xq, c1, true, 32 * it + threadIdx.x / VPR, threadIdx.x % VPR * V);
  if (CLAMP && top > kHalfMax) atomicOr(&a.ws.hdr->status, 1);
  __syncthreads();
  // gate A^T[j rows, k lanes] of source tile jt and key tile kt from their product, as operands with the key on the lanes
  auto gate = [&](acc_t& aT, frag<T> (&fa)[2], int jt, int kt) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) aT[r] = fast_rcp(1.f + fast_exp2(aT[r]));
    if (jt == kt) {   // j > k only
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (acc_row(r, g) <= c) aT[r] = 0.f;
    }
    fa[0] = chain<T>(aT, 0);
    fa[1] = chain<T>(aT, 1);
  };
  // ---- scores of key tile kt: source tiles of one parity per wave ----------------------------------------------------------
  const int kt = wave % kShortTiles, half = wave / kShortTiles, i = 32 * it + c;
  acc_t su;   // [k rows, i lanes]
  zero(su);
  // (loops, not copies: the code runs once a launch, and is waited for)
  if (kt <= it) {
    float large = 0.f;
#pragma clang loop unroll(disable)
    for (int jt = kt + half; jt <= it; jt += 2) {
      acc_t aT, t;   // gate [j rows, k lanes], T' [j rows, i lanes]
      zero(aT);
      zero(t);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        mma(aT, ld_nat<T>(s_ku, LD, 32 * jt + c, 16 * ks + 8 * g), ld_nat<T>(s_qu, LD, 32 * kt + c, 16 * ks + 8 * g));
        mma(t, ld_nat<T>(s_vu, LD, 32 * jt + c, 16 * ks + 8 * g), ld_nat<T>(s_qc, LD, c, 16 * ks + 8 * g));
      }
      frag<T> fa[2];
      gate(aT, fa, jt, kt);
      if constexpr (__is_same(T, fp16_t)) {   // T' beyond the fp16 range is clamped, and reported
        float m = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) m = fmaxf(m, fabsf(t[r]));
        large = fmaxf(large, m);
        if (__builtin_amdgcn_ballot_w64(m > kHalfMax) != 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) t[r] = __builtin_amdgcn_fmed3f(t[r], -kHalfMax, kHalfMax);
        }
      }
      if (jt == it) {   // j <= i
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (acc_row(r, g) > c) t[r] = 0.f;
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) mma(su, fa[s2], chain<T>(t, s2));
    }
    if (large > kHalfMax) atomicOr(&a.ws.hdr->status, 2);
    settle();
    if (half == 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s_sum[(kt * 16 + r) * 64 + lane] = su[r];
    }
  }
  // ---- lookahead keys of key tile `it`: by wave a source tile, summed in the order of the waves ---------------------------------
  acc_t u[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(u[nt]);
  const int jt = it + wave - kShortTiles;   // (the upper waves)
  if (want_u && half == 1 && jt < tiles) {
    acc_t aT;
    zero(aT);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) mma(aT, ld_nat<T>(s_ku, LD, 32 * jt + c, 16 * ks + 8 * g), ld_nat<T>(s_qu, LD, 32 * it + c, 16 * ks + 8 * g));
    frag<T> fa[2];
    gate(aT, fa, jt, it);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mma(u[nt], ld_free<T, true>(s_vu + 32 * jt * LD, LD, 32 * nt, HD, 16 * s2, c, g), fa[s2]);
  }
  settle();
  __syncthreads();
  acc_t o[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(o[nt]);
  float m = kLowest, l = 0.f;
  if (half == 0 && kt <= it) {
    acc_t sc;
    zero(sc);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) mma(sc, ld_nat<T>(s_kc, LD, 32 * kt + c, 16 * ks + 8 * g), ld_nat<T>(s_qc, LD, c, 16 * ks + 8 * g));
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float sut = (su[r] + s_sum[(kt * 16 + r) * 64 + lane]) * su_mul;
      const float sg = fast_rcp(1.f + fast_exp2(-sut));
      sc[r] = __builtin_fmaf(-sut, sg, sc[r]);
    }
    if (kt == it) {   // causal
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (acc_row(r, g) > c) sc[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) m = fmaxf(m, sc[r]);
    m = fmaxf(m, __shfl_xor(m, 32));
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sc[r] = fast_exp2(sc[r] - m);
      l += sc[r];
    }
    l += __shfl_xor(l, 32);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const frag<T> fp = chain<T>(sc, s2);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mma(o[nt], ld_free<T, true>(s_vc + 32 * kt * LD, LD, 32 * nt, HD, 16 * s2, c, g), fp);
    }
  }
  // ---- the key tiles --------------------------------------------------------------------------------------------------------
  float *const s_part = reinterpret_cast<float*>(castle_smem), *const s_stat = s_part + kShortTiles * 64 * NT * 16;
  settle();
  __syncthreads();   // operands and score sums are read
  if (half == 0) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) s_part[((kt * NT + nt) * 16 + r) * 64 + lane] = o[nt][r];
    s_stat[(2 * kt) * 64 + lane] = m;
    s_stat[(2 * kt + 1) * 64 + lane] = l;
  }
  __syncthreads();
  if (half == 0 && i < L) {   // wave w: every fourth quad of a row
    float w[kShortTiles], M = kLowest, sum = 0.f;
#pragma unroll
    for (int k = 0; k < kShortTiles; ++k) M = fmaxf(M, s_stat[(2 * k) * 64 + lane]);
#pragma unroll
    for (int k = 0; k < kShortTiles; ++k) {
      w[k] = fast_exp2(s_stat[(2 * k) * 64 + lane] - M);
      sum = __builtin_fmaf(w[k], s_stat[(2 * k + 1) * 64 + lane], sum);
    }
    const float inv = 1.f / sum;
    TI* dst = head_ptr_mut<TI>(a.out, b, h) + (int64_t)i * a.out.sl;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = 32 * nt + 8 * kt + 4 * g;
      vec<float, 4> v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < kShortTiles; ++k)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(w[k] * inv, s_part[((k * NT + nt) * 16 + 4 * kt + e) * 64 + lane], v[e]);
      if (n < HD) st4<TI>(dst + n, __builtin_convertvector(v, vec<TI, 4>));
    }
  }
  if (!want_u) return;
  __syncthreads();
  if (half == 1) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) s_part[((kt * NT + nt) * 16 + r) * 64 + lane] = u[nt][r];
  }
  __syncthreads();
  if (half == 0 && i < L) {
    TI* dst = head_ptr_mut<TI>(a.U, b, h) + (int64_t)i * a.U.sl;
    const bool half_format = a.u_half != 0;
    const float mul = half_format ? su_mul * kUHalfScale : su_mul;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = 32 * nt + 8 * kt + 4 * g;
      vec<float, 4> v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int k = 0; k < kShortTiles; ++k) v[e] += s_part[((k * NT + nt) * 16 + 4 * kt + e) * 64 + lane];
        v[e] *= mul;
        if (half_format) v[e] = __builtin_amdgcn_fmed3f(v[e], -kHalfMax, kHalfMax);
      }
      if (n < HD) {
        if (half_format) st4<fp16_t>(reinterpret_cast<fp16_t*>(dst + n), __builtin_convertvector(v, vec<fp16_t, 4>));
        else st4<TI>(dst + n, __builtin_convertvector(v, vec<TI, 4>));
      }
    }
  }
}

__global__ void clear_status_kernel(int* status) { *status = 0; }

// 1: not for this shape.  Every workgroup converts all rows up to its tile's: beyond two tiles that pays while the workgroups are in flight together,
// up to three to a CU.  General / here, us: 128 rows x 128 heads (512 workgroups), d = 64 26.9 / 21.8; 96 x 256 (768) 33.9 / 28.0, d = 16 20.1 / 10.7;
// 128 x 256 (1024) 37.0 / 39.5, d = 32 with 1024 heads 61.7 / 61.7; 64 x 4096, two tiles, 389 / 119.
constexpr int kShortGroups = 3 * 256;
int launch_short(const FwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream) {
  const int tiles = (a.s.L + 31) / 32;
  if (dtype == 0 || tiles > kShortTiles || (tiles > 2 && a.s.B * a.s.H > kShortGroups / tiles)) return 1;
  return by_type16(dtype, bf16_operands, [&](auto t, auto ti) {
    using T = decltype(t); using TI = decltype(ti);
    return by_head_dim<T>(a.s.d, [&](auto hd) {
      constexpr int HD = decltype(hd)::value;
      const int lds = short_lds<T, HD>(tiles);
      if (lds > kMaxLds - 1024) return 1;
      if (!a.amax_ready) hipLaunchKernelGGL(clear_status_kernel, dim3(1), dim3(1), 0, stream, &a.ws.hdr->status);
      auto go = [&](auto kernel, PerDeviceOnce& once) {
        bool& configured = once.flag();
        if (!configured) configured = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kMaxLds - 1024) == hipSuccess;
        if (!configured) return false;
        ProfScope ps(kSlotAttn, stream);
        hipLaunchKernelGGL(kernel, dim3(a.s.B * a.s.H * tiles), dim3(kShortThreads), lds, stream, a);
        return true;
      };
      static PerDeviceOnce plain, rotary;
      if (!(a.s.rotary ? go(&short_kernel<T, TI, HD, true>, rotary) : go(&short_kernel<T, TI, HD, false>, plain))) return -3;
      return hipGetLastError() == hipSuccess ? 0 : -3;
    });
  });
}

}  // namespace castle
