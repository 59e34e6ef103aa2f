// CASTLE backward kernels over 32-row work items with independent waves: see castle_narrow.hip.
#include "castle_narrow_tiles.h"

namespace castle {

// ---------------------------------------------------------------------------
// shared rows of the keys (-c1 Qu, Kc, Vc); two operand tiles and a tile of T' rows per wave
// and the row sums of a block (-log2 normaliser, -delta)
template <typename T, int HD> constexpr int key_narrow_wave_bytes() { return 2 * wave_tile_bytes<T, HD>() + t_tile_bytes<T>() + 2 * kNB * 4; }
template <typename T, int HD, int W> constexpr int key_narrow_lds() {
  return 3 * wave_tile_bytes<T, HD>() + max2(W * key_narrow_wave_bytes<T, HD>(), reduce_bytes<HD, W>());
}

template <typename T, typename TI, int HD, int W>
__global__ __launch_bounds__(64 * W, (narrow_waves<T, HD>())) void key_narrow_kernel(BwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>(), LD = lds_ld_tr<T>(HD), LDT = kLdT64<T>;
  constexpr bool SB = sizeof(T) == 4 || HD >= 64;   // scalar bases where the registers are short (d = 32, 32 heads x 777: 41.9 us without, 43.8 with)
  constexpr bool STAGES = sizeof(T) == 2 && HD == 64;   // two waves per SIMD just fit
  const int L = a.s.L, BH = a.s.B * a.s.H, nblk = (L + kNB - 1) / kNB;
  int kt, bh;   // key tile 0 meets every query
  narrow_item<T, HD>(BH, (L + 31) / 32, a.s.cus, kt, bh);
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const float c0 = a.s.scale, c1 = a.s.scale * kLog2e;
  const float su_mul = a.ws.hdr->su_mul, gun = a.bhdr->grad_unscale;
  const int kw0 = 32 * kt, k = kw0 + c, Iw = kt >> 1;
  T* s_qu = reinterpret_cast<T*>(castle_smem);
  T* s_kc = s_qu + 32 * LD;
  T* s_vc = s_kc + 32 * LD;
  unsigned char* work = castle_smem + 3 * wave_tile_bytes<T, HD>();
  T* s_a = reinterpret_cast<T*>(work + wave * key_narrow_wave_bytes<T, HD>());
  T* s_b = s_a + 32 * LD;
  T* s_t = s_b + 32 * LD;
  float* s_sum = reinterpret_cast<float*>(s_t + 32 * LDT);
  float* red = reinterpret_cast<float*>(work);
  const T* qc = prep_ptr<T>(a.ws.qc_p, bh, a.s.Lp, HD);
  const T* ku = prep_ptr<T>(a.ws.ku_p, bh, a.s.Lp, HD);
  const T* vu = prep_ptr<T>(a.ws.vu_p, bh, a.s.Lp, HD);
  const T* dout = prep_ptr<T>(a.dout_p, bh, a.s.Lp, HD);
  const T* tb = reinterpret_cast<const T*>(a.ws.t_blk) + (int64_t)bh * a.s.Lp * kNB;
  const T* ttb = reinterpret_cast<const T*>(a.ws.tt_blk) + (int64_t)bh * a.s.Lp * kNB;
  const T* usnap = reinterpret_cast<const T*>(a.ws.usnap) + (int64_t)bh * snap_rows(a.s.nblk) * HD;
  T* gsnap = reinterpret_cast<T*>(a.gsnap) + (int64_t)bh * snap_rows(a.s.nblk) * HD;
  // dS / dSu tiles of these keys: element (key k, chained slot) of query tile it at it * 1024 + s2 * 512 + k * 16 + g * 8
  const int64_t tile0 = (int64_t)bh * a.s.Lp * a.s.Lp + (int64_t)kt * (a.s.Lp / 32) * 1024;
  const uint32_t tile_at = (c * 16 + g * 8) * (int)sizeof(T);
  T* ds_mat = reinterpret_cast<T*>(a.ds_mat) + tile0;
  T* dsu_mat = reinterpret_cast<T*>(a.dsu_mat) + tile0;
  const float* lse = a.ws.lse + (int64_t)bh * a.s.Lp;
  const float* delta = a.delta + (int64_t)bh * a.s.Lp;

  for (int t = wave; t < 3; t += W) {
    Flat32<T, HD, SB> f;
    f.load(prep_ptr<T>(t == 0 ? a.ws.qu_p : t == 1 ? a.ws.kc_p : a.ws.vc_p, bh, a.s.Lp, HD) + (int64_t)kw0 * HD);
    f.store(s_qu + t * 32 * LD, t == 0 ? -c1 : 1.f);
  }
  const int seg = (nblk - Iw + W - 1) / W;
  // both gates of a block side by side, so that one chain of products fills the wait for the other (key pass of 16 heads x 1000 rows, d = 64: 41.5 -> 39.3 us);
  // at d = 128, one wave to a SIMD, without room for a second tile of sources on its way, 3 % slower; fp32 was not tried
  constexpr bool PAIRED = sizeof(T) == 2 && HD <= 64;
  const int lo = min(nblk, Iw + wave * seg), hi = min(nblk, lo + seg);
  // Edges need no branches: rows beyond the sequence are zero and have lse = inf, sources and queries in front of
  // the keys are masked; such tiles give zeros (and the tile arrays have room for them).
  // gate A^T[j rows, k lanes] of source tile jt from the product of its Ku rows
  auto gate_of = [&](acc_t& aT, int jt) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 16; ++r) aT[r] = fast_rcp(1.f + fast_exp2(aT[r]));
    if (jt <= kt) {   // j > k only
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * (jt - kt) + acc_row(r, g) <= c) aT[r] = 0.f;
    }
  };
  auto gate = [&](acc_t& aT, int jt) __attribute__((always_inline)) {   // whose Ku rows are in s_a
    zero(aT);
#pragma unroll
    for (int s = 0; s < KS; ++s) mma(aT, ld_nat<T>(s_a, LD, c, 16 * s + 8 * g), ld_nat<T>(s_qu, LD, c, 16 * s + 8 * g));
    gate_of(aT, jt);
  };
  // the next tiles, requested one step ahead
  Flat32<T, HD, SB> pa, pb;
  Flat32<T, kNB, SB> pt;

  acc_t G[NT];   // [n rows, k lanes]
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(G[nt]);
  {
    // ---- pass A: score chain, dVc, dKc, this part's contribution to the reverse state -------------------------------
    acc_t dvc[NT], dkc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) { zero(dvc[nt]); zero(dkc[nt]); }
    // one row of the block per lane, a block ahead: loaded where a tile needs them, they were waited for twice a block
    // (12 heads x 1000 rows: 50.9 -> 48.1 us)
    float nl = 0.f, nd = 0.f;
    auto sums = [&](int I) __attribute__((always_inline)) {
      nl = load_at<float, SB>(lse + I * kNB, 4 * lane);
      nd = load_at<float, SB>(delta + I * kNB, 4 * lane);
    };
    if (lo < hi) {
      pa.load(ku + (int64_t)lo * kNB * HD);
      if (PAIRED) pb.load(ku + ((int64_t)lo * kNB + 32) * HD);
      sums(lo);
    }
    __syncthreads();   // the shared rows are there
    for (int I = lo; I < hi; ++I) {
      const bool there = I * kNB + lane < L;
      s_sum[lane] = there ? -nl * kLog2e : -INFINITY;
      s_sum[kNB + lane] = there ? -nd : 0.f;
      sums(min(I + 1, nblk - 1));
      frag<T> fub[KS], fa[2][2];
      load_snap32<T, HD>(fub, I > Iw ? usnap + (usnap_off(I) + kw0) * HD : ku, c, g);
      if constexpr (PAIRED) {
        wave_lds_order<STAGES>();
        pa.store(s_a);
        pb.store(s_b);
        wave_lds_order<STAGES>();
        pa.load(qc + (int64_t)I * kNB * HD);
        pb.load(dout + (int64_t)I * kNB * HD);
        pt.load(tb + (int64_t)I * kNB * kNB);
        acc_t a0, a1;
        zero(a0);
        zero(a1);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const frag<T> fq = ld_nat<T>(s_qu, LD, c, 16 * s + 8 * g);
          mma(a0, ld_nat<T>(s_a, LD, c, 16 * s + 8 * g), fq);
          mma(a1, ld_nat<T>(s_b, LD, c, 16 * s + 8 * g), fq);
        }
        gate_of(a0, 2 * I);
        gate_of(a1, 2 * I + 1);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          fa[0][s2] = chain<T>(a0, s2);
          fa[1][s2] = chain<T>(a1, s2);
        }
      } else {
#pragma unroll
        for (int jtl = 0; jtl < 2; ++jtl) {
          wave_lds_order<STAGES>();
          pa.store(s_a);
          wave_lds_order<STAGES>();
          if (jtl == 0) {
            pa.load(ku + ((int64_t)I * kNB + 32) * HD);
          } else {
            pa.load(qc + (int64_t)I * kNB * HD);
            pb.load(dout + (int64_t)I * kNB * HD);
            pt.load(tb + (int64_t)I * kNB * kNB);
          }
          acc_t aT;
          gate(aT, 2 * I + jtl);
          fa[jtl][0] = chain<T>(aT, 0);
          fa[jtl][1] = chain<T>(aT, 1);
        }
      }
      if (I == Iw) {   // no state in front of the keys' own block
#pragma unroll
        for (int s = 0; s < KS; ++s) fub[s] = zero_frag<T>();
      }
#pragma unroll
      for (int itl = 0; itl < 2; ++itl) {
        const int it = 2 * I + itl;
        acc_t sc, su, dp;   // [i rows, k lanes]; sc starts from -lse, dp from -delta of its row
        zero(su);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const vec<float, 4> l4 = *reinterpret_cast<const vec<float, 4>*>(s_sum + 32 * itl + 8 * q + 4 * g);
          const vec<float, 4> d4 = *reinterpret_cast<const vec<float, 4>*>(s_sum + kNB + 32 * itl + 8 * q + 4 * g);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            sc[4 * q + e] = l4[e];
            dp[4 * q + e] = d4[e];
          }
        }
        wave_lds_order<STAGES>();
        pa.store(s_a);
        pb.store(s_b);
        pt.store(s_t);
        wave_lds_order<STAGES>();
        if (itl == 0) {
          pa.load(qc + ((int64_t)I * kNB + 32) * HD);
          pb.load(dout + ((int64_t)I * kNB + 32) * HD);
          if (!STAGES) pt.load(tb + ((int64_t)I * kNB + 32) * kNB);
        } else {
          pa.load(ku + (int64_t)min(I + 1, nblk - 1) * kNB * HD);
          if (PAIRED) pb.load(ku + ((int64_t)min(I + 1, nblk - 1) * kNB + 32) * HD);
        }
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const frag<T> oq = ld_nat<T>(s_a, LD, c, 16 * s + 8 * g);
          mma(su, oq, fub[s]);
          mma(sc, oq, ld_nat<T>(s_kc, LD, c, 16 * s + 8 * g));
          mma(dp, ld_nat<T>(s_b, LD, c, 16 * s + 8 * g), ld_nat<T>(s_vc, LD, c, 16 * s + 8 * g));
        }
#pragma unroll
        for (int jt = 0; jt < 2; ++jt)
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2)
            if (jt <= itl) mma(su, ld_chain<T>(s_t, LDT, c, 32 * jt + 16 * s2, g), fa[jt][s2]);
        if (it <= kt) {   // queries before the key see nothing
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (32 * (it - kt) + acc_row(r, g) < c) sc[r] = -INFINITY;
        }
        acc_t ds, dsu;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float sut = su[r] * su_mul;                             // log2(e) * Su
          const float sg = fast_rcp(1.f + fast_exp2(-sut));
          const float p = fast_exp2(__builtin_fmaf(-sut, sg, sc[r]));   // sc carries -lse
          const float dsv = p * dp[r];                                  // dp carries -delta
          const float y = sut * kLn2;                                   // true Su
          const float t = __builtin_fmaf(-y, sg, y);                    // y (1 - sigmoid)
          const float sp = __builtin_fmaf(sg, t, sg);                   // silu'(y)
          sc[r] = p;
          ds[r] = dsv;
          dsu[r] = -dsv * sp * su_mul;
        }
        // (requested with the other two it is what does not fit the registers, and a spilled piece is waited for on the spot: 3 x 4 heads of 1000
        // rows, layer with its gradients 186 -> 179 us, with the scalar bases)
        if (STAGES && itl == 0) pt.load(tb + ((int64_t)I * kNB + 32) * kNB);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          const frag<T> fp = chain<T>(sc, s2), fds = chain<T>(ds, s2), fdsu = chain<T>(dsu, s2);
          store_at<frag_mem<T>, SB>(ds_mat + (int64_t)it * 1024 + s2 * 512, tile_at, fds);   // whole lines per store
          store_at<frag_mem<T>, SB>(dsu_mat + (int64_t)it * 1024 + s2 * 512, tile_at, fdsu);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) {
            const frag<T> qt = ld_free<T, true>(s_a, LD, 32 * nt, HD, 16 * s2, c, g);
            mma(dvc[nt], ld_free<T, true>(s_b, LD, 32 * nt, HD, 16 * s2, c, g), fp);
            mma(dkc[nt], qt, fds);
            mma(G[nt], qt, fdsu);
          }
        }
      }
    }
    TI* row = head_ptr_mut<TI>(a.dkc, b, h) + (int64_t)k * a.dkc.sl;
    reduce_waves<W, NT>(red, dkc, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
      if (k < L) store_quad<TI, HD>(row, 32 * nt + 8 * q + 4 * g, v, kLn2 * gun, a.s.rotary ? k : -1);
    });
    row = head_ptr_mut<TI>(a.dvc, b, h) + (int64_t)k * a.dvc.sl;
    reduce_waves<W, NT>(red, dvc, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
      if (k < L) store_quad<TI, HD>(row, 32 * nt + 8 * q + 4 * g, v, gun, -1);
    });
  }
  // ---- the reverse state behind this wave's part: the sum over the later parts --------------------------------------
  settle();
  __syncthreads();
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[((wave * NT + nt) * 16 + r) * 64 + lane] = G[nt][r];
  __syncthreads();
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float sum = 0.f;
#pragma unroll
      for (int w = 1; w < W; ++w) sum = __builtin_fmaf(w > wave ? 1.f : 0.f, red[((w * NT + nt) * 16 + r) * 64 + lane], sum);
      G[nt][r] = sum;
    }
  __syncthreads();   // the memory holds tiles again
  // ---- pass B: from the last block of the part down ------------------------------------------------------------------
  acc_t dqu[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(dqu[nt]);
  auto request = [&](int I, int jtl) __attribute__((always_inline)) {   // the source tile 2 I + jtl
    const int64_t r = (int64_t)I * kNB + 32 * jtl;
    pa.load(ku + r * HD);
    pb.load(vu + r * HD);
    pt.load(ttb + r * kNB);
  };
  if (lo < hi) request(hi - 1, 0);
  for (int I = hi - 1; I >= lo; --I) {
    frag<T> fdsu[2][2];   // this wave stored them in pass A
#pragma unroll
    for (int itl = 0; itl < 2; ++itl)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) fdsu[itl][s2] = load_at<frag_mem<T>, SB>(dsu_mat + (int64_t)(2 * I + itl) * 1024 + s2 * 512, tile_at);
    settle();
    if (I <= nblk - 2) store_snap_tile<T, HD, NT>(gsnap + (gsnap_off(I) + kw0) * HD, G, c, g);
#pragma unroll
    for (int jtl = 0; jtl < 2; ++jtl) {
      wave_lds_order<STAGES>();
      pa.store(s_a);
      pb.store(s_b);
      pt.store(s_t);
      wave_lds_order<STAGES>();
      if (jtl == 0) {
        request(I, 1);
      } else {
        pa.load(qc + (int64_t)I * kNB * HD);
        pb.load(qc + ((int64_t)I * kNB + 32) * HD);
      }
      acc_t aT, dA;   // [j rows, k lanes]
      gate(aT, 2 * I + jtl);
      zero(dA);
#pragma unroll
      for (int s = 0; s < KS; ++s) mma(dA, ld_chain<T>(s_b, LD, c, 16 * s, g), chain<T>(G[s / 2], s % 2));
#pragma unroll
      for (int itl = 0; itl < 2; ++itl)
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2)
          if (itl >= jtl) mma(dA, ld_chain<T>(s_t, LDT, c, 32 * itl + 16 * s2, g), fdsu[itl][s2]);
#pragma unroll
      for (int r = 0; r < 16; ++r) dA[r] *= __builtin_fmaf(-aT[r], aT[r], aT[r]);   // dZ = dA A (1 - A)
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const frag<T> fdz = chain<T>(dA, s2);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) mma(dqu[nt], ld_free<T, true>(s_a, LD, 32 * nt, HD, 16 * s2, c, g), fdz);
      }
    }
    // the block joins the reverse state
    wave_lds_order<STAGES>();
    pa.store(s_a);
    pb.store(s_b);
    wave_lds_order<STAGES>();
    request(max(I - 1, 0), 0);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        mma(G[nt], ld_free<T, true>(s_a, LD, 32 * nt, HD, 16 * s2, c, g), fdsu[0][s2]);
        mma(G[nt], ld_free<T, true>(s_b, LD, 32 * nt, HD, 16 * s2, c, g), fdsu[1][s2]);
      }
  }
  TI* row = head_ptr_mut<TI>(a.dqu, b, h) + (int64_t)k * a.dqu.sl;
  reduce_waves<W, NT>(red, dqu, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    if (k < L) store_quad<TI, HD>(row, 32 * nt + 8 * q + 4 * g, v, c0 * kLn2 * gun, a.s.rotary ? k : -1);
  });
}

// ---------------------------------------------------------------------------
template <typename T, int HD> constexpr int query_narrow_wave_bytes() { return 2 * wave_tile_bytes<T, HD>() + 2 * (int)sizeof(T) * 32 * kLdX<T>; }
template <typename T, int HD, int W> constexpr int query_narrow_lds() {
  return 3 * wave_tile_bytes<T, HD>() + t_tile_bytes<T>() + max2(W * query_narrow_wave_bytes<T, HD>(), reduce_bytes<HD, W>());
}

template <typename T, typename TI, int HD, int W>
__global__ __launch_bounds__(64 * W, (narrow_waves<T, HD>())) void query_narrow_kernel(BwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>(), LD = lds_ld_tr<T>(HD), LDX = kLdX<T>;
  constexpr bool SB = sizeof(T) == 4 || HD >= 64;   // scalar bases where the registers are short (d = 32, 32 heads x 777: 28.7 us without, 29.5 with)
  constexpr bool STAGES = sizeof(T) == 2;   // d = 64: 13 spilled registers, none in the loop
  const int L = a.s.L, BH = a.s.B * a.s.H, ntile = (L + 31) / 32, nblk = (L + kNB - 1) / kNB;
  int rank, bh;
  narrow_item<T, HD>(BH, ntile, a.s.cus, rank, bh);
  const int it = ntile - 1 - rank;   // the last rows meet the most keys
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const float c0 = a.s.scale, c1 = a.s.scale * kLog2e;
  const float gun = a.bhdr->grad_unscale, vu_scale = a.ws.hdr->vu_scale;
  const int i = 32 * it + c, I = it >> 1, half = it & 1;
  const bool has_g = I <= nblk - 2;                     // a reverse state exists behind the block
  const bool next = half == 0 && it + 1 < ntile;        // the block's second tile of queries exists and is not this one
  // the rows of the tile as sources (-c1 Ku, Vu) and, for a second tile, the -c1 Ku rows of the block's first one, whose
  // sources its queries meet too; shared by the waves
  T* s_ku = reinterpret_cast<T*>(castle_smem);
  T* s_vu = s_ku + 32 * LD;
  T* s_k0 = s_vu + 32 * LD;
  T* s_tt = s_k0 + 32 * LD;   // T'^T rows of the tile
  unsigned char* work = castle_smem + 3 * wave_tile_bytes<T, HD>() + t_tile_bytes<T>();
  T* s_x = reinterpret_cast<T*>(work + wave * query_narrow_wave_bytes<T, HD>());
  T* s_y = s_x + 32 * LD;
  T* s_ds = s_y + 32 * LD;
  T* s_dsu = s_ds + 32 * LDX;
  float* red = reinterpret_cast<float*>(work);
  const T* qc = prep_ptr<T>(a.ws.qc_p, bh, a.s.Lp, HD);
  const T* kc = prep_ptr<T>(a.ws.kc_p, bh, a.s.Lp, HD);
  const T* qu = prep_ptr<T>(a.ws.qu_p, bh, a.s.Lp, HD);
  const T* ku = prep_ptr<T>(a.ws.ku_p, bh, a.s.Lp, HD);
  const T* vu = prep_ptr<T>(a.ws.vu_p, bh, a.s.Lp, HD);
  const T* ttb = reinterpret_cast<const T*>(a.ws.tt_blk) + (int64_t)bh * a.s.Lp * kNB;
  const T* usnap = reinterpret_cast<const T*>(a.ws.usnap) + (int64_t)bh * snap_rows(a.s.nblk) * HD + usnap_off(I) * HD;
  const T* gsnap = reinterpret_cast<const T*>(a.gsnap) + (int64_t)bh * snap_rows(a.s.nblk) * HD + (has_g ? gsnap_off(I) * HD : 0);
  const T* ds_mat = reinterpret_cast<const T*>(a.ds_mat) + (int64_t)bh * a.s.Lp * a.s.Lp + (int64_t)it * 1024;
  const T* dsu_mat = reinterpret_cast<const T*>(a.dsu_mat) + (int64_t)bh * a.s.Lp * a.s.Lp + (int64_t)it * 1024;
  const uint32_t tile_at = (c * 16 + g * 8) * (int)sizeof(T);
  const int64_t tile_row = (int64_t)(a.s.Lp / 32) * 1024;   // between the tiles of consecutive key tiles

  for (int t = wave; t < 4; t += W) {
    if (t < 3) {
      Flat32<T, HD, SB> f;
      f.load(t == 0 ? ku + (int64_t)it * 32 * HD : t == 1 ? vu + (int64_t)it * 32 * HD : ku + (int64_t)I * kNB * HD);
      f.store(s_ku + t * 32 * LD, t == 1 ? 1.f : -c1);
    } else {
      Flat32<T, kNB, SB> f;
      f.load(ttb + (int64_t)it * 32 * kNB);
      f.store(s_tt);
    }
  }
  __syncthreads();
  acc_t dqc[NT], dku[NT], dvu[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) { zero(dqc[nt]); zero(dku[nt]); zero(dvu[nt]); }
  // dT[i, j] = sum over keys of dSu[i, k] A[k, j] inside the block.  own: [j rows, i lanes], both of this tile.  far: a
  // first tile as the sources of the second tile's queries, [i rows, j lanes]; a second tile as the queries of the first
  // tile's sources, [j rows, i lanes].
  acc_t own, far;
  zero(own);
  zero(far);

  // What a key tile begins with is requested at the end of the one before, where registers get free (Kc and the state: in the
  // middle of their own): 8 heads x 2000 rows 58.3 -> 55.0 us, 2 x 3000 71.7 -> 67.5.  Not with one wave per SIMD (d = 128
  // 72.6 -> 84, fp32 118 -> 122: the registers then move between the two files).
  constexpr bool EARLY = narrow_waves<T, HD>() == 2;
  Flat32<T, HD, SB> pq;
  frag<T> og[KS], fds[2], fdsu[2], fdsn[2];
  auto request = [&](int kt) __attribute__((always_inline)) {
    pq.load(qu + (int64_t)kt * 32 * HD);
    load_snap32<T, HD>(og, has_g ? gsnap + (int64_t)kt * 32 * HD : kc, c, g);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      fds[s2] = load_at<frag_mem<T>, SB>(ds_mat + kt * tile_row + s2 * 512, tile_at);
      fdsu[s2] = load_at<frag_mem<T>, SB>(dsu_mat + kt * tile_row + s2 * 512, tile_at);
      if constexpr (EARLY) fdsn[s2] = load_at<frag_mem<T>, SB>(dsu_mat + kt * tile_row + (next ? 1024 : 0) + s2 * 512, tile_at);
      else fdsn[s2] = next ? load_at<frag_mem<T>, SB>(dsu_mat + kt * tile_row + 1024 + s2 * 512, tile_at) : zero_frag<T>();
    }
  };
  if constexpr (EARLY) request(min(wave, it));
  for (int kt = wave; kt <= it; kt += W) {
    const int Kb = kt >> 1;
    if constexpr (!EARLY) request(kt);
    Flat32<T, HD, SB> pk;
    frag<T> ou[KS];
    if (EARLY && !next) {
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) fdsn[s2] = zero_frag<T>();
    }
    wave_lds_order<STAGES>();
    pq.store(s_x);
    wave_lds_order<STAGES>();
    // gates A[k rows, j lanes] of the own sources, and of the first tile's sources for a second tile (zero where they do
    // not lie behind the keys)
    acc_t aK, a0;
    zero(aK);
    zero(a0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const frag<T> oq = ld_nat<T>(s_x, LD, c, 16 * s + 8 * g);
      mma(a0, oq, ld_nat<T>(s_k0, LD, c, 16 * s + 8 * g));
      mma(aK, oq, ld_nat<T>(s_ku, LD, c, 16 * s + 8 * g));
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      aK[r] = fast_rcp(1.f + fast_exp2(aK[r]));
      a0[r] = fast_rcp(1.f + fast_exp2(a0[r]));
    }
    if (kt + 1 >= it) {   // j > k only
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (c + 32 * (it - kt) <= acc_row(r, g)) aK[r] = 0.f;
        if (c + 32 * (2 * I - kt) <= acc_row(r, g)) a0[r] = 0.f;
      }
    }
    frag<T> fa[2], f0[2];
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) { fa[s2] = chain<T>(aK, s2); f0[s2] = chain<T>(a0, s2); }
    if (!has_g) {
#pragma unroll
      for (int s = 0; s < KS; ++s) og[s] = zero_frag<T>();
    }
    put_rows32<T, HD>(s_y, og, c, g);
    // the tiles in natural query order, [key][query], to be read with the query on the lanes
    auto put_tile = [&](T* tile, const frag<T> (&f)[2]) __attribute__((always_inline)) {
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        vec<T, 4> lo, hi;
#pragma unroll
        for (int e = 0; e < 4; ++e) { lo[e] = f[s2][e]; hi[e] = f[s2][4 + e]; }
        st4<T>(tile + c * LDX + 16 * s2 + 4 * g, lo);
        st4<T>(tile + c * LDX + 16 * s2 + 4 * g + 8, hi);
      }
    };
    put_tile(s_dsu, fdsu);
    put_tile(s_ds, fdsn);
    wave_lds_order<STAGES>();
    frag<T> bdsu[2];
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      bdsu[s2] = ld_free<T, true>(s_dsu, LDX, 0, 32, 16 * s2, c, g);
      const frag<T> bdsn = ld_free<T, true>(s_ds, LDX, 0, 32, 16 * s2, c, g);
      mma(own, fa[s2], bdsu[s2]);
      // one of the two products, chosen by operands: the second tile of the block, or the first (zeros without a second)
      mma(far, half == 1 ? f0[s2] : bdsn, half == 1 ? bdsu[s2] : fa[s2]);
    }
    wave_lds_order<STAGES>();
    put_tile(s_ds, fds);
    pk.load(kc + (int64_t)kt * 32 * HD);
    load_snap32<T, HD>(ou, Kb < I ? usnap + (int64_t)kt * 32 * HD : kc, c, g);
    // dA = dSu^T T' + G' Vu^T, dZ, dKu, dVu
    acc_t dA;
    zero(dA);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      mma(dA, fdsu[s2], ld_chain<T>(s_tt, kLdT64<T>, c, 32 * half + 16 * s2, g));
      mma(dA, fdsn[s2], ld_chain<T>(s_tt, kLdT64<T>, c, 32 + 16 * s2, g));   // (zeros without a next tile)
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) mma(dA, og[s], ld_nat<T>(s_vu, LD, c, 16 * s + 8 * g));
#pragma unroll
    for (int r = 0; r < 16; ++r) dA[r] *= __builtin_fmaf(-aK[r], aK[r], aK[r]);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const frag<T> fdz = chain<T>(dA, s2);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        mma(dku[nt], ld_free<T, true>(s_x, LD, 32 * nt, HD, 16 * s2, c, g), fdz);
        mma(dvu[nt], ld_free<T, true>(s_y, LD, 32 * nt, HD, 16 * s2, c, g), fa[s2]);
      }
    }
    wave_lds_order<STAGES>();
    if constexpr (EARLY) request(min(kt + W, it));   // unconditional: the last iteration repeats a tile
    if (Kb >= I) {
#pragma unroll
      for (int s = 0; s < KS; ++s) ou[s] = zero_frag<T>();
    }
    pk.store(s_x);
    put_rows32<T, HD>(s_y, ou, c, g);
    wave_lds_order<STAGES>();
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const frag<T> bds = ld_free<T, true>(s_ds, LDX, 0, 32, 16 * s2, c, g);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        mma(dqc[nt], ld_free<T, true>(s_x, LD, 32 * nt, HD, 16 * s2, c, g), bds);
        mma(dqc[nt], ld_free<T, true>(s_y, LD, 32 * nt, HD, 16 * s2, c, g), bdsu[s2]);
      }
    }
  }
  // ---- epilogue: dT inside the block:  dqc += dT Vu,  dvu += dT^T Qc' ---------------------------------------------------
  total_of_waves<W>(red, own, wave, lane);
  total_of_waves<W>(red, far, wave, lane);
  __syncthreads();   // the memory holds tiles again
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if (acc_row(r, g) > c) own[r] = 0.f;   // j <= i
  // the own tile with i as the contraction: X[i][j]
#pragma unroll
  for (int q = 0; q < 4; ++q) st4<T>(s_ds + c * LDX + 8 * q + 4 * g, pack4<T>(own, q));
  // the Qc' rows of the tile; a second tile: the first tile's Vu rows (for dqc), a first tile: the second tile's Qc' rows
  Flat32<T, HD, SB> pi, pk;
  pi.load(qc + (int64_t)it * 32 * HD);
  pk.load(half == 1 ? vu + (int64_t)I * kNB * HD : qc + (int64_t)min(it + 1, a.s.Lp / 32 - 1) * 32 * HD);
  pi.store(s_y);
  pk.store(s_x);
  wave_lds_order<STAGES>();
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (nt % W != wave) continue;   // every column tile once
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const frag<T> x = ld_free<T, true>(s_x, LD, 32 * nt, HD, 16 * s2, c, g), ff = chain<T>(far, s2);
      mma(dqc[nt], x, half == 1 ? ff : zero_frag<T>());
      mma(dvu[nt], x, half == 1 ? zero_frag<T>() : ff);
      mma(dqc[nt], ld_free<T, true>(s_vu, LD, 32 * nt, HD, 16 * s2, c, g), chain<T>(own, s2));
      mma(dvu[nt], ld_free<T, true>(s_y, LD, 32 * nt, HD, 16 * s2, c, g), ld_free<T, true>(s_ds, LDX, 0, 32, 16 * s2, c, g));
    }
  }
  const int pos = a.s.rotary ? i : -1;
  TI* row = head_ptr_mut<TI>(a.dqc, b, h) + (int64_t)i * a.dqc.sl;
  reduce_waves<W, NT>(red, dqc, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    if (i < L) store_quad<TI, HD>(row, 32 * nt + 8 * q + 4 * g, v, c0 * gun, pos);
  });
  row = head_ptr_mut<TI>(a.dku, b, h) + (int64_t)i * a.dku.sl;
  reduce_waves<W, NT>(red, dku, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    if (i < L) store_quad<TI, HD>(row, 32 * nt + 8 * q + 4 * g, v, c0 * kLn2 * gun, pos);
  });
  row = head_ptr_mut<TI>(a.dvu, b, h) + (int64_t)i * a.dvu.sl;
  reduce_waves<W, NT>(red, dvu, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    if (i < L) store_quad<TI, HD>(row, 32 * nt + 8 * q + 4 * g, v, kLn2 * gun * vu_scale, pos);
  });
}

// ---------------------------------------------------------------------------
template <typename T, typename TI, int HD, int W> static int bwd_narrow(const BwdArgs& a, hipStream_t stream) {   // W: waves of the key kernel
  constexpr int key_lds = key_narrow_lds<T, HD, W>(), query_lds = query_narrow_lds<T, HD, 4>();
  static_assert(key_lds <= kMaxLds && query_lds <= kMaxLds);
  static PerDeviceOnce once;
  bool& configured = once.flag();
  if (!configured) configured = raise_lds(&key_narrow_kernel<T, TI, HD, W>, key_lds) && raise_lds(&query_narrow_kernel<T, TI, HD, 4>, query_lds);
  if (!configured) return -3;
  const dim3 grid((a.s.L + 31) / 32 * a.s.B * a.s.H);
  {
    ProfScope ps(kSlotBwdKey, stream);
    hipLaunchKernelGGL((key_narrow_kernel<T, TI, HD, W>), grid, dim3(64 * W), key_lds, stream, a);
  }
  {
    ProfScope ps(kSlotBwdQuery, stream);
    hipLaunchKernelGGL((query_narrow_kernel<T, TI, HD, 4>), grid, dim3(256), query_lds, stream, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
int launch_bwd_narrow(const BwdArgs& a, int dtype, bool bf16_operands, hipStream_t stream) {
  return by_type(dtype, bf16_operands, [&](auto t, auto ti) {
    using T = decltype(t); using TI = decltype(ti);
    return by_head_dim<T>(a.s.d, [&](auto hd) {
      constexpr int HD = decltype(hd)::value;
      if constexpr (narrow_waves<T, HD>() == 2)
        if (eight_waves<T, HD>(a.s)) return bwd_narrow<T, TI, HD, 8>(a, stream);
      return bwd_narrow<T, TI, HD, 4>(a, stream);
    });
  });
}

}  // namespace castle
