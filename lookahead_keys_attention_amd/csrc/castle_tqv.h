// The T' blocks of a forward pass (see tqv_block): run by the trailing workgroups of both scan launches.
#pragma once
#include "castle_tiles.h"
#include "castle_params.h"

namespace castle {

// T' of one 64-row block, by the four waves of a workgroup (one 32x32 tile each).  These blocks have
// no kernel of their own: they are the last workgroups of the scan launch, which reads none of them,
// so they run in the slots the scan's tail leaves empty (its last fifth runs at under half occupancy:
// the launch cannot end before the 64-block sweep of key group 0 does).
template <typename T, typename TI, int HD>
__device__ __forceinline__ void tqv_block(const FwdArgs& a, int I, int bh) {
  constexpr int KS = HD / 16;
  constexpr int TB = kNB / 32;
  static_assert(TB * TB == kThreads / 64, "one 32x32 tile of the block per wave");
  const int lane = lane_id(), c = lane & 31, g = lane >> 5;
  const T* qc = prep_ptr<T>(a.ws.qc_p, bh, a.s.Lp, HD);   // pre-scaled by c1
  const T* vu = prep_ptr<T>(a.ws.vu_p, bh, a.s.Lp, HD);
  T* tb = reinterpret_cast<T*>(a.ws.t_blk) + (int64_t)bh * a.s.Lp * kNB;
  T* ttb = reinterpret_cast<T*>(a.ws.tt_blk) + (int64_t)bh * a.s.Lp * kNB;
  T* ttx = reinterpret_cast<T*>(a.ws.ttx_blk) + (int64_t)bh * a.s.Lp * kNB;
  const int it = wave_id() / TB, jt = wave_id() % TB;
  const int64_t i = (int64_t)I * kNB + 32 * it + c;   // A-operand row
  const int64_t j = (int64_t)I * kNB + 32 * jt + c;   // B-operand row
  // cross quarter of a pair of blocks, (Qc'_{I+1} Vu_I^T)^T for even I: same sources, the queries
  // of the next block, no mask (every query is later).  All operand loads are issued together.
  const bool cross = (I & 1) == 0 && I + 1 < a.s.nblk;
  frag<T> fq[KS], fv[KS], fx[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    fq[s] = ldg_nat<T>(qc, HD, i, 16 * s + 8 * g, true);
    fv[s] = ldg_nat<T>(vu, HD, j, 16 * s + 8 * g, true);
    fx[s] = ldg_nat<T>(qc, HD, i + kNB, 16 * s + 8 * g, cross);
  }
  acc_t acc, accx;
  zero(acc);
  zero(accx);
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    mma(acc, fq[s], fv[s]);
    mma(accx, fx[s], fv[s]);
  }
  if constexpr (__is_same(T, fp16_t)) {   // T' beyond the fp16 range is clamped (and reported in the header)
    bool clamped = false;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float y = __builtin_amdgcn_fmed3f(acc[r], -kHalfMax, kHalfMax), yx = __builtin_amdgcn_fmed3f(accx[r], -kHalfMax, kHalfMax);
      clamped |= (y != acc[r] && acc[r] == acc[r]) || (yx != accx[r] && accx[r] == accx[r]);
      acc[r] = y;
      accx[r] = yx;
    }
    if (clamped) atomicOr(&a.ws.hdr->status, 2);
  }
  // acc[r] = (Qc' Vu^T)[il = 32 it + acc_row][jl = 32 jt + c]; stored as T' = tril(.)
  const int jl = 32 * jt + c;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int il = 32 * it + acc_row(r, g);
    acc[r] = jl > il ? 0.f : acc[r];
    tb[((int64_t)I * kNB + il) * kNB + jl] = (T)acc[r];
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    st4<T>(ttb + ((int64_t)I * kNB + jl) * kNB + 32 * it + 8 * q + 4 * g, pack4<T>(acc, q));
  if (cross) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      st4<T>(ttx + ((int64_t)I * kNB + jl) * kNB + 32 * it + 8 * q + 4 * g, pack4<T>(accx, q));
  }
}

}  // namespace castle
