// CASTLE forward and backward kernels over 32-row work items with independent waves ("narrow" kernels).
//
// The kernels of castle_fwd.hip / castle_bwd.hip give 128 rows to a workgroup and walk the sequence in one serial
// chain per workgroup: right when there are hundreds of such workgroups per launch, a tenth of the chip when a batch
// has a dozen heads of a thousand tokens, and at one wave per SIMD with idle matrix pipes for fp32, whose matrix
// instructions take eight times as long as the data movement the wide tiles save.  Here a workgroup owns 32 rows and its
// W waves share the walk: every wave takes its own part of the keys (or queries), nothing is exchanged inside the loops
// (no barriers), and the partial results meet once at the end, in fp32 through LDS.  Every operand tile is copied as whole
// lines into LDS that belongs to one wave, while the tile before it is worked on; the rows of the workgroup itself are
// in LDS once, for all waves.  What bounds them is the wait for those tiles, two waves per SIMD at most (one at d = 128 and
// fp32), and for fp32 the matrix instructions: operator forward and backward at 2 x 8 heads of 1024 rows 1426 -> 431 us
// in fp32; 8 x 4 heads of 777 rows at d = 32 in fp16 269 -> 116 us (with the host path measured; the kernels took 193
// of it and take 136 with the small kernels around them).
//
//   scan_narrow    32 keys; the waves split the source blocks: every wave sums its own part first, then sweeps it
//                  again from the sum of the parts before it, storing the snapshots (two gates per pair instead
//                  of one, a chain of 2 / W of the blocks)
//   attn_narrow    32 queries; wave w takes the key tiles w, w + W, ..: own online softmax, merged at the end
//   key_narrow     32 keys; the waves split the query blocks: pass A forms P, dS, dSu of the part (dVc, dKc, the part's
//                  contribution to the reverse state, and the dS / dSu tiles for the next kernel), pass B walks the
//                  part again from the reverse state behind it (gsnap, dA, dZ, dQu)
//   query_narrow   32 rows as queries and as lookahead sources; wave w takes the key tiles w, w + W, ..: dQc, dKu,
//                  dVu, dT
// Branches behind matrix instructions: nothing between the last MFMA on an accumulator and the first ordinary read of it
// may be skipped by a branch.  Where such a branch jumps over a run of loads, the compiler (ROCm 7.2) counts the
// loads as waiting time on both ways, and on the taken one the first registers are read before they are written
// (seen in the scan at d = 128: three accumulator registers of the last tile).  So the loads of a next tile are
// unconditional (the last iteration repeats a tile), and conditional products come before unconditional ones.  Where sums over
// waves or stores follow a loop of products, settle() stands in front of the first read; not where a barrier and reads of
// LDS stand between anyway (the weights of the attention's partial results), nor where nothing can be skipped (a snapshot
// at the top of the next iteration).
//
// Definitions, units and range control are those of castle_fwd.hip and castle_bwd.hip.  Rows beyond the sequence are
// not visited (only what a partly filled tile of 32 holds).
//
// The backward kernels are in castle_narrow_bwd.hip, compiled by themselves: the compiler keeps the results of matrix instructions in vector registers here
// (d = 128: scan 23.3 -> 21.9 us, attn 31.3 -> 28.2, 8 heads x 1000 rows), which the key kernel at d = 128 has no room for (55.3 -> 67.1, spills).
#include "castle_narrow_tiles.h"

namespace castle {

// ---------------------------------------------------------------------------
template <typename T, int HD, int W> constexpr int scan_narrow_lds() { return max2((2 * W + 1) * wave_tile_bytes<T, HD>(), reduce_bytes<HD, W>()); }

template <typename T, typename TI, int HD, int W>
__global__ __launch_bounds__(64 * W, (narrow_waves<T, HD>())) void scan_narrow_kernel(FwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>(), LD = lds_ld_tr<T>(HD);
  // every tile of the padded length: the backward kernels of either kind read the snapshots this leaves
  const int L = a.s.L, BH = a.s.B * a.s.H, ntile = a.s.Lp / 32, nblk = a.s.nblk;
  {
    const int n_scan = ntile * BH;
    if ((int)blockIdx.x >= n_scan) {   // behind the key tiles: the T' blocks
      const int id = blockIdx.x - n_scan;
      if (wave_id() < 4) tqv_block<T, TI, HD>(a, id / BH, id % BH);
      return;
    }
  }
  int kt, bh;   // key tile 0 sweeps every source block
  narrow_item<T, HD>(BH, ntile, a.s.cus, kt, bh);
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const float c1 = a.s.scale * kLog2e;
  const int kw0 = 32 * kt, k = kw0 + c, Kb = kt >> 1;
  T* s_ku = reinterpret_cast<T*>(castle_smem + wave * 2 * wave_tile_bytes<T, HD>());
  T* s_vu = s_ku + 32 * LD;
  T* s_qu = reinterpret_cast<T*>(castle_smem + W * 2 * wave_tile_bytes<T, HD>());
  const T* qu = prep_ptr<T>(a.ws.qu_p, bh, a.s.Lp, HD);
  const T* ku = prep_ptr<T>(a.ws.ku_p, bh, a.s.Lp, HD);
  const T* vu = prep_ptr<T>(a.ws.vu_p, bh, a.s.Lp, HD);
  T* snap = reinterpret_cast<T*>(a.ws.usnap) + (int64_t)bh * snap_rows(a.s.nblk) * HD;

  frag<T> fq[KS];   // -c1 Qu rows of the keys
  if (wave == 0) {
    Flat32<T, HD, HD >= 64> f;
    f.load(qu + (int64_t)kw0 * HD);
    f.store(s_qu, -c1);
  }
  __syncthreads();
#pragma unroll
  for (int s = 0; s < KS; ++s) fq[s] = ld_nat<T>(s_qu, LD, c, 16 * s + 8 * g);
  acc_t st[NT];   // state^T: rows n, columns k
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(st[nt]);

  const int seg = (nblk - Kb + W - 1) / W;
  const int lo = min(nblk, Kb + wave * seg), hi = min(nblk, lo + seg);
  auto sweep = [&](bool keep) __attribute__((always_inline)) {
    // source tiles of 32 rows, two per block; the rows of the next one are requested while one is worked on
    const int first = max(2 * lo, kt), last = min(2 * hi, ntile);
    Flat32<T, HD, HD >= 64> pk, pv;
    if (first < last) {
      pk.load(ku + (int64_t)first * 32 * HD);
      pv.load(vu + (int64_t)first * 32 * HD);
    }
    for (int jt = first; jt < last; ++jt) {
      const int I = jt >> 1;
      if (keep && I > Kb && (jt == first || !(jt & 1))) store_snap_tile<T, HD, NT>(snap + (usnap_off(I) + kw0) * HD, st, c, g);
      wave_lds_order<>();
      pk.store(s_ku);
      pv.store(s_vu);
      wave_lds_order<>();
      const int nx = min(jt + 1, last - 1);   // (no branch here: see the note on branches behind matrix instructions)
      pk.load(ku + (int64_t)nx * 32 * HD);
      pv.load(vu + (int64_t)nx * 32 * HD);
      acc_t aT;   // A^T: rows j, columns k
      zero(aT);
#pragma unroll
      for (int s = 0; s < KS; ++s) mma(aT, ld_nat<T>(s_ku, LD, c, 16 * s + 8 * g), fq[s]);
#pragma unroll
      for (int r = 0; r < 16; ++r) aT[r] = fast_rcp(1.f + fast_exp2(aT[r]));
      if (jt == kt) {   // j > k only
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (acc_row(r, g) <= c) aT[r] = 0.f;
      }
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const frag<T> fa = chain<T>(aT, s2);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) mma(st[nt], ld_free<T, true>(s_vu, LD, 32 * nt, HD, 16 * s2, c, g), fa);
      }
    }
  };
  if (seg < nblk - Kb) {   // more than one part: the sums of the parts in front of this wave's
    if (hi < nblk) sweep(false);
    float* red = reinterpret_cast<float*>(castle_smem);
    settle();
    __syncthreads();   // the tiles are dead
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) red[((wave * NT + nt) * 16 + r) * 64 + lane] = st[nt][r];
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < W - 1; ++w) sum = __builtin_fmaf(w < wave ? 1.f : 0.f, red[((w * NT + nt) * 16 + r) * 64 + lane], sum);
        st[nt][r] = sum;
      }
    __syncthreads();   // the memory holds tiles again
  }
  if (lo >= hi) return;
  sweep(true);
  settle();
  if (hi == nblk && a.U.ptr != nullptr && k < L) {
    TI* dst = head_ptr_mut<TI>(a.U, b, h) + (int64_t)k * a.U.sl;
    const float su_mul = a.ws.hdr->su_mul;   // the state was built from vu * vu_scale
    bool half_format = false;
    if constexpr (sizeof(TI) == 2) half_format = a.u_half != 0;
    const float mul = half_format ? su_mul * kUHalfScale : su_mul;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        st[nt][r] *= mul;
        if (half_format) st[nt][r] = __builtin_amdgcn_fmed3f(st[nt][r], -kHalfMax, kHalfMax);
      }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = 32 * nt + 8 * q + 4 * g;
        if (n < HD) {
          if (half_format) st4<fp16_t>(reinterpret_cast<fp16_t*>(dst + n), pack4<fp16_t>(st[nt], q));
          else st4<TI>(dst + n, pack4<TI>(st[nt], q));
        }
      }
  }
}

// ---------------------------------------------------------------------------
// shared rows (Qc', two tiles of Ku, T'), three tiles per wave; the merge reuses all of it
template <typename T, int HD, int W> constexpr int attn_narrow_tiles() { return max2((3 + 3 * W) * wave_tile_bytes<T, HD>() + t_tile_bytes<T>(), reduce_bytes<HD, W>()); }
template <typename T, int HD, int W> constexpr int attn_narrow_lds() { return attn_narrow_tiles<T, HD, W>() + W * 64 * 8; }

template <typename T, typename TI, int HD, int W>
__global__ __launch_bounds__(64 * W, (narrow_waves<T, HD>())) void attn_narrow_kernel(FwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>(), LD = lds_ld_tr<T>(HD);
  const int L = a.s.L, BH = a.s.B * a.s.H, ntile = (L + 31) / 32;
  int rank, bh;
  narrow_item<T, HD>(BH, ntile, a.s.cus, rank, bh);
  const int it = ntile - 1 - rank;   // the last queries see the most keys
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const float c1 = a.s.scale * kLog2e;
  const float su_mul = a.ws.hdr->su_mul;
  const int i = 32 * it + c, I = it >> 1, half = it & 1;
  T* s_rows = reinterpret_cast<T*>(castle_smem);   // Qc' rows of the tile, -c1 Ku rows of the block's two tiles
  T* s_t = s_rows + 3 * 32 * LD;                   // T' rows of the tile
  T* s_q = reinterpret_cast<T*>(castle_smem + (3 + 3 * wave) * wave_tile_bytes<T, HD>() + t_tile_bytes<T>());
  T* s_k = s_q + 32 * LD;
  T* s_v = s_k + 32 * LD;
  float* s_stat = reinterpret_cast<float*>(castle_smem + attn_narrow_tiles<T, HD, W>());
  const T* qc = prep_ptr<T>(a.ws.qc_p, bh, a.s.Lp, HD);   // pre-scaled by c1
  const T* kc = prep_ptr<T>(a.ws.kc_p, bh, a.s.Lp, HD);
  const T* vc = prep_ptr<T>(a.ws.vc_p, bh, a.s.Lp, HD);
  const T* qu = prep_ptr<T>(a.ws.qu_p, bh, a.s.Lp, HD);
  const T* ku = prep_ptr<T>(a.ws.ku_p, bh, a.s.Lp, HD);
  const T* tb = reinterpret_cast<const T*>(a.ws.t_blk) + (int64_t)bh * a.s.Lp * kNB;
  const T* snap = reinterpret_cast<const T*>(a.ws.usnap) + (int64_t)bh * snap_rows(a.s.nblk) * HD + usnap_off(I) * HD;

  for (int t = wave; t < 4; t += W) {
    if (t < 3) {
      Flat32<T, HD, HD >= 64> f;
      f.load(t == 0 ? qc + (int64_t)it * 32 * HD : ku + ((int64_t)I * kNB + 32 * (t - 1)) * HD);
      f.store(s_rows + t * 32 * LD, t == 0 ? 1.f : -c1);
    } else {
      Flat32<T, kNB, HD >= 64> f;
      f.load(tb + (int64_t)it * 32 * kNB);
      f.store(s_t);
    }
  }
  __syncthreads();
  frag<T> fqc[KS], fku[2][KS], ft[2][2];   // c1 Qc rows, -c1 Ku rows of the block, T' rows (chained order)
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    fqc[s] = ld_nat<T>(s_rows, LD, c, 16 * s + 8 * g);
#pragma unroll
    for (int jt = 0; jt < 2; ++jt) fku[jt][s] = ld_nat<T>(s_rows + (1 + jt) * 32 * LD, LD, c, 16 * s + 8 * g);
  }
#pragma unroll
  for (int jt = 0; jt < 2; ++jt)
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) ft[jt][s2] = ld_chain<T>(s_t, kLdT64<T>, c, 32 * jt + 16 * s2, g);   // (zero where j > i)
  acc_t o[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(o[nt]);
  float m = -INFINITY, l = 0.f;

  Flat32<T, HD, HD >= 64> pq, pk, pv;
  frag<T> nu[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) nu[s] = zero_frag<T>();
  if (wave <= it) {
    pq.load(qu + (int64_t)wave * 32 * HD);
    pk.load(kc + (int64_t)wave * 32 * HD);
    pv.load(vc + (int64_t)wave * 32 * HD);
    if ((wave >> 1) < I) load_snap32<T, HD>(nu, snap + (int64_t)wave * 32 * HD, c, g);
  }
  for (int kt = wave; kt <= it; kt += W) {
    const int nx = min(kt + W, it);   // the loads of the next tile are unconditional: the last iteration repeats one
    wave_lds_order<>();
    pq.store(s_q);
    pk.store(s_k);
    pv.store(s_v);
    wave_lds_order<>();
    pq.load(qu + (int64_t)nx * 32 * HD);
    pk.load(kc + (int64_t)nx * 32 * HD);
    pv.load(vc + (int64_t)nx * 32 * HD);
    if ((kt >> 1) >= I) {   // keys of the own block: no state yet
#pragma unroll
      for (int s = 0; s < KS; ++s) nu[s] = zero_frag<T>();
    }
    // gates of the block's sources up to this tile: A^T[j rows, k lanes], used as the operand with k on the lanes
    frag<T> fa[2][2];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt) {
      if (jt <= half && 2 * I + jt >= kt) {
        acc_t aT;
        zero(aT);
#pragma unroll
        for (int s = 0; s < KS; ++s) mma(aT, fku[jt][s], ld_nat<T>(s_q, LD, c, 16 * s + 8 * g));
#pragma unroll
        for (int r = 0; r < 16; ++r) aT[r] = fast_rcp(1.f + fast_exp2(aT[r]));
        if (2 * I + jt == kt) {   // j > k only
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (acc_row(r, g) <= c) aT[r] = 0.f;
        }
        fa[jt][0] = chain<T>(aT, 0);
        fa[jt][1] = chain<T>(aT, 1);
      } else {
        fa[jt][0] = zero_frag<T>();
        fa[jt][1] = zero_frag<T>();
      }
    }
    acc_t sc, su;   // [k rows, i lanes]
    zero(sc);
    zero(su);
    if (half) {
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) mma(su, fa[1][s2], ft[1][s2]);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      mma(su, nu[s], fqc[s]);
      mma(sc, ld_nat<T>(s_k, LD, c, 16 * s + 8 * g), fqc[s]);
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) mma(su, fa[0][s2], ft[0][s2]);
    load_snap32<T, HD>(nu, (nx >> 1) < I ? snap + (int64_t)nx * 32 * HD : kc, c, g);
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float sut = su[r] * su_mul;
      const float sg = fast_rcp(1.f + fast_exp2(-sut));
      sc[r] = __builtin_fmaf(-sut, sg, sc[r]);
    }
    if (kt == it) {   // causal mask
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (acc_row(r, g) > c) sc[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {
      const float m_new = fmaxf(m, mx), alpha = fast_exp2(m - m_new);
      l *= alpha;
      m = m_new;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[nt][r] *= alpha;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sc[r] = fast_exp2(sc[r] - m);
      l += sc[r];
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const frag<T> fp = chain<T>(sc, s2);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) mma(o[nt], ld_free<T, true>(s_v, LD, 32 * nt, HD, 16 * s2, c, g), fp);
    }
  }
  // merge the waves: common maximum, then weighted sums
  l += __shfl_xor(l, 32);
  s_stat[(wave * 64 + lane) * 2] = m;
  s_stat[(wave * 64 + lane) * 2 + 1] = l;
  __syncthreads();
  float M = -INFINITY, lt = 0.f;
#pragma unroll
  for (int w = 0; w < W; ++w) M = fmaxf(M, s_stat[(w * 64 + lane) * 2]);
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const float mw = s_stat[(w * 64 + lane) * 2];
    lt += mw == -INFINITY ? 0.f : fast_exp2(mw - M) * s_stat[(w * 64 + lane) * 2 + 1];
  }
  const float wt = m == -INFINITY ? 0.f : fast_exp2(m - M) / lt;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[nt][r] *= wt;
  TI* dst = head_ptr_mut<TI>(a.out, b, h) + (int64_t)i * a.out.sl;
  reduce_waves<W, NT>(reinterpret_cast<float*>(castle_smem), o, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    const int n = 32 * nt + 8 * q + 4 * g;
    if (i < L && n < HD) st4<TI>(dst + n, __builtin_convertvector(v, vec<TI, 4>));
  });
  if (wave == 0 && g == 0 && i < L) a.ws.lse[(int64_t)bh * a.s.Lp + i] = (M + __builtin_log2f(lt)) * kLn2;
}

// ---------------------------------------------------------------------------
template <typename T, typename TI, int HD, int W> static int scan_narrow(const FwdArgs& a, hipStream_t stream) {
  constexpr int lds = scan_narrow_lds<T, HD, W>();
  static_assert(lds <= kMaxLds);
  static PerDeviceOnce once;
  bool& configured = once.flag();
  if (!configured) configured = raise_lds(&scan_narrow_kernel<T, TI, HD, W>, lds);
  if (!configured) return -3;
  const int BH = a.s.B * a.s.H;
  ProfScope ps(kSlotScan, stream);
  hipLaunchKernelGGL((scan_narrow_kernel<T, TI, HD, W>), dim3(a.s.Lp / 32 * BH + (a.with_t ? a.s.nblk * BH : 0)), dim3(64 * W), lds, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
template <typename T, typename TI, int HD, int W> static int attn_narrow(const FwdArgs& a, hipStream_t stream) {
  constexpr int lds = attn_narrow_lds<T, HD, W>();
  static_assert(lds <= kMaxLds);
  static PerDeviceOnce once;
  bool& configured = once.flag();
  if (!configured) configured = raise_lds(&attn_narrow_kernel<T, TI, HD, W>, lds);
  if (!configured) return -3;
  ProfScope ps(kSlotAttn, stream);
  hipLaunchKernelGGL((attn_narrow_kernel<T, TI, HD, W>), dim3((a.s.L + 31) / 32 * a.s.B * a.s.H), dim3(64 * W), lds, stream, a);
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
int launch_scan_narrow(const FwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream) {
  return by_type(dtype, bf16_operands, [&](auto t, auto ti) {
    using T = decltype(t); using TI = decltype(ti);
    return by_head_dim<T>(a.s.d, [&](auto hd) {
      constexpr int HD = decltype(hd)::value;
      if constexpr (narrow_waves<T, HD>() == 2)
        if (eight_waves<T, HD>(a.s)) return scan_narrow<T, TI, HD, 8>(a, stream);
      return scan_narrow<T, TI, HD, 4>(a, stream);
    });
  });
}
int launch_attn_narrow(const FwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream) {
  return by_type(dtype, bf16_operands, [&](auto t, auto ti) {
    using T = decltype(t); using TI = decltype(ti);
    return by_head_dim<T>(a.s.d, [&](auto hd) {
      constexpr int HD = decltype(hd)::value;
      if constexpr (narrow_waves<T, HD>() == 2)
        if (eight_waves<T, HD>(a.s)) return attn_narrow<T, TI, HD, 8>(a, stream);
      return attn_narrow<T, TI, HD, 4>(a, stream);
    });
  });
}

}  // namespace castle
