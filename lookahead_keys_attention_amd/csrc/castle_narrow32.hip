// CASTLE forward and backward kernels of fp32 tensors: the 32-row work items of castle_narrow.hip (its comments on the split of the work, on
// branches behind matrix instructions and on edges hold here too) on pairs of fp16 numbers (castle_split.h).
//
// What bounds them is no longer the matrix instructions (busy 17-19 % of the time; 55-60 % when they were the fp32 ones) but waiting: for LDS, for the tiles a wave
// requests one step ahead, for the end of chains of matrix instructions.  Two waves per SIMD where the registers allow it (prefix sums, attention); the
// backward kernels need 450 registers, and with 256 and eight waves, without anything requested ahead, they spill (key 105 -> 157 us, query 76 -> 180).
// 2 x 8 heads x 1024 rows, d = 64, us, fp32 instructions / here: scan 59 / 29, attention 75 / 36, key 161 / 103, query 113 / 76.
//
// Everything these kernels pass on to each other is stored as such pairs, split once, with what they are to be multiplied with: operand copies, T'
// blocks, snapshots of both states, dS / dSu tiles.
#include "castle_tiles.h"
#include "castle_params.h"
#include "castle_profile.h"
#include "castle_split.h"
#include "castle_waves.h"
#include "castle_dispatch.h"
#include "castle_narrow.h"

namespace castle {

extern __shared__ __attribute__((aligned(16))) unsigned char castle_smem[];

constexpr int kW = 4;   // waves of a workgroup
template <int HD> constexpr int kTile = split_tile_bytes<HD>();   // bytes of a padded LDS tile
template <int HD> constexpr int kTileElems = 2 * split_plane<HD>();

// A snapshot tile.  f: accumulator tiles in chained order (rows n, key c on the lanes)
template <int HD> __device__ __forceinline__ void store_snap_halves(fp16_t* tile, const split8 (&f)[narrow_nt<HD>() * 2], int c, int g) {
#pragma unroll
  for (int s = 0; s < HD / 16; ++s)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      vec<fp16_t, 4> h, l;
#pragma unroll
      for (int e = 0; e < 4; ++e) { h[e] = f[s].h[4 * q + e]; l[e] = f[s].l[4 * q + e]; }
      const int n = 16 * s + 8 * q + 4 * g;
      st4_stream<fp16_t>(tile + snap_elem<fp16_t>(c, n), h);
      st4_stream<fp16_t>(tile + 32 * HD + snap_elem<fp16_t>(c, n), l);
    }
}

// ---------------------------------------------------------------------------
// A wave copies a tile: blockIdx.z selects the operand.  Bound by memory and launch: 25 MB in and out 10.9 us.
template <int HD>
__global__ __launch_bounds__(64 * kW, 4) void prep_split_kernel(FwdArgs a) {
  constexpr int N = HD / 16, VPR = HD / 8;
  const int bh = blockIdx.y, b = bh / a.s.H, h = bh % a.s.H, tiles = a.s.Lp / 32, tile = blockIdx.x * kW + wave_id();
  View4 src;
  void* dst;
  float mul = 1.f;
  switch (blockIdx.z) {
    case kOpQc: src = a.qc; dst = a.ws.qc_p; mul = a.s.scale * kLog2e; break;
    case kOpKc: src = a.kc; dst = a.ws.kc_p; break;
    case kOpVc: src = a.vc; dst = a.ws.vc_p; break;
    case kOpQu: src = a.qu; dst = a.ws.qu_p; break;
    case kOpKu: src = a.ku; dst = a.ws.ku_p; break;
    default: src = a.vu; dst = a.ws.vu_p; break;
  }
  if (blockIdx.x == 0 && bh == 0 && blockIdx.z == 0 && threadIdx.x == 0) {
    a.ws.hdr->status = 0;
    a.ws.hdr->vu_scale = 1.f;
    a.ws.hdr->su_mul = 1.f;
  }
  const float* from = head_ptr<float>(src, b, h) + (32 * (int64_t)tile + lane_id() / VPR) * src.sl + lane_id() % VPR * 8;
  const int64_t step = 64 / VPR * src.sl;
  vec<float, 8> x[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    x[n] = zero_frag<float>();
    if (32 * tile + lane_id() / VPR + n * (64 / VPR) < a.s.L) x[n] = *reinterpret_cast<const frag_mem<float>*>(from + n * step);
  }
  if (a.s.rotary && blockIdx.z != kOpVc) {   // every operand but Vc is rotated by its position
#pragma unroll
    for (int n = 0; n < N; ++n) {
      const float row = (float)(32 * tile + lane_id() / VPR + n * (64 / VPR));
#pragma unroll
      for (int e = 0; e < 4; ++e) CASTLE_ROPE_PAIR(x[n][2 * e], x[n][2 * e + 1], row, lane_id() % VPR * 4 + e, HD, false);
    }
  }
#pragma unroll
  for (int n = 0; n < N; ++n) x[n] *= mul;
  const float inv = store_split_tile<HD>(reinterpret_cast<fp16_t*>(dst) + ((int64_t)bh * tiles + tile) * split_elems<HD>(), x);
  if (lane_id() == 0) a.ws.op_mul[((int64_t)blockIdx.z * gridDim.y + bh) * tiles + tile] = inv;
}

// ---------------------------------------------------------------------------
// T' = tril(Qc'_I Vu_I^T) of a block of 64 rows and its transpose, one 32 x 32 tile per wave: trailing workgroups of the scan launch.  Both are formed as
// products, in the order in which they become operands: no transposition, whole lines per store.
template <int HD> __device__ __forceinline__ void t_block_split(const FwdArgs& a, int I, int bh) {
  constexpr int KS = HD / 16;
  const int lane = lane_id(), c = lane & 31, g = lane >> 5, BH = a.s.B * a.s.H, tiles = a.s.Lp / 32;
  const int it = wave_id() >> 1, jt = wave_id() & 1;
  SplitRows<HD> fq, fv;
  fq.load(split_tiles<HD>(a.ws.qc_p, bh, tiles) + (2 * I + it) * split_elems<HD>());
  fv.load(split_tiles<HD>(a.ws.vu_p, bh, tiles) + (2 * I + jt) * split_elems<HD>());
  const float mul = a.ws.op_mul[((int64_t)kOpQc * BH + bh) * tiles + 2 * I + it] * a.ws.op_mul[((int64_t)kOpVu * BH + bh) * tiles + 2 * I + jt];
  acc_t t, tt;   // [j rows, i lanes], [i rows, j lanes]
  zero(t);
  zero(tt);
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    mma(t, fv.f[s], fq.f[s]);
    mma(tt, fq.f[s], fv.f[s]);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    t[r] = 32 * jt + acc_row(r, g) > 32 * it + c ? 0.f : t[r] * mul;
    tt[r] = 32 * jt + c > 32 * it + acc_row(r, g) ? 0.f : tt[r] * mul;
  }
  uint32_t* s_max = reinterpret_cast<uint32_t*>(castle_smem);
  const uint32_t bits = wave_max_bits(abs_max(t));
  if (lane == 0) s_max[wave_id()] = bits;
  __syncthreads();
  const TileScale ts = tile_scale(max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3])));
  if (threadIdx.x == 0) a.ws.t_mul[(int64_t)bh * a.s.nblk + I] = ts.inv;
  // tiles of 32 rows: their fragments in chained order
  fp16_t* tb = split_tiles_mut<kNB>(a.ws.t_blk, bh, tiles) + (2 * I + it) * split_elems<kNB>() + 8 * lane;
  fp16_t* ttb = split_tiles_mut<kNB>(a.ws.tt_blk, bh, tiles) + (2 * I + jt) * split_elems<kNB>() + 8 * lane;
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) {
    const split8 f = chain_split(t, s2, ts.mul), ft = chain_split(tt, s2, ts.mul);
    *reinterpret_cast<frag_mem<fp16_t>*>(tb + 512 * (2 * jt + s2)) = f.h;
    *reinterpret_cast<frag_mem<fp16_t>*>(tb + 512 * (4 + 2 * jt + s2)) = f.l;
    *reinterpret_cast<frag_mem<fp16_t>*>(ttb + 512 * (2 * it + s2)) = ft.h;
    *reinterpret_cast<frag_mem<fp16_t>*>(ttb + 512 * (4 + 2 * it + s2)) = ft.l;
  }
}

// Ku comes as fragments, only Vu passes through LDS, to be read by columns.  (Both through LDS 35 us; split on their way, from fp32 copies, 41; two key tiles a wave,
// which halves what a CU draws from L2, 54: half as many waves to wait.)
template <int HD> constexpr int scan_split_lds() { return max2(kW * kTile<HD>, reduce_bytes<HD, kW>()); }

template <int HD>
__global__ __launch_bounds__(64 * kW, 2) void scan_split_kernel(FwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>(), E = split_elems<HD>();
  const int L = a.s.L, BH = a.s.B * a.s.H, nblk = a.s.nblk, tiles = a.s.Lp / 32;
  {
    const int n_scan = tiles * BH;
    if ((int)blockIdx.x >= n_scan) {   // behind the key tiles: the T' blocks
      const int id = blockIdx.x - n_scan;
      t_block_split<HD>(a, id / BH, id % BH);
      return;
    }
  }
  int kt, bh;   // key tile 0 sweeps every source block
  work_item_snake(BH, tiles, a.s.cus, kt, bh);
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const int kw0 = 32 * kt, k = kw0 + c, Kb = kt >> 1;
  fp16_t* s_vu = reinterpret_cast<fp16_t*>(castle_smem + wave * kTile<HD>);
  const fp16_t* qu = split_tiles<HD>(a.ws.qu_p, bh, tiles);
  const fp16_t* ku = split_tiles<HD>(a.ws.ku_p, bh, tiles);
  const fp16_t* vu = split_tiles<HD>(a.ws.vu_p, bh, tiles);
  const float* m_ku = a.ws.op_mul + ((int64_t)kOpKu * BH + bh) * tiles;
  const float* m_vu = a.ws.op_mul + ((int64_t)kOpVu * BH + bh) * tiles;
  fp16_t* snap = reinterpret_cast<fp16_t*>(a.ws.usnap) + (int64_t)bh * snap_rows(nblk) * 2 * HD;
  float* u_mul = a.ws.u_mul + (int64_t)bh * nblk * tiles + kt;
  const float z0 = -a.s.scale * kLog2e * a.ws.op_mul[((int64_t)kOpQu * BH + bh) * tiles + kt];

  SplitRows<HD> fq;   // Qu rows of the keys
  fq.load(qu + kt * E);
  acc_t st[NT];   // state^T: rows n, columns k
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(st[nt]);

  const int seg = (nblk - Kb + kW - 1) / kW;
  const int lo = min(nblk, Kb + wave * seg), hi = min(nblk, lo + seg);
  auto sweep = [&](bool keep) __attribute__((always_inline)) {
    const int first = max(2 * lo, kt), last = 2 * hi;
    SplitRows<HD> pk, pv;
    float mk = 0.f, mv = 0.f;
    if (first < last) {
      pk.load(ku + first * E);
      pv.load(vu + first * E);
      mk = m_ku[first];
      mv = m_vu[first];
    }
    for (int jt = first; jt < last; ++jt) {
      const int I = jt >> 1;
      if (keep && I > Kb && !(jt & 1)) {
        float m = 0.f;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) m = abs_max(st[nt], m);
        const TileScale us = tile_scale(wave_max_bits(m));
        split8 f[2 * NT];
#pragma unroll
        for (int s = 0; s < 2 * NT; ++s) f[s] = chain_split(st[s / 2], s % 2, us.mul);
        store_snap_halves<HD>(snap + (usnap_off(I) + kw0) * 2 * HD, f, c, g);
        if (lane == 0) u_mul[(int64_t)I * tiles] = us.inv;
      }
      wave_lds_order<>();
      pv.store(s_vu);
      wave_lds_order<>();
      const int nx = min(jt + 1, last - 1);   // (no branch: the last iteration repeats a tile)
      pv.load(vu + nx * E);
      const float z = z0 * mk, v_mul = mv * kUnitInv;
      mk = m_ku[nx];
      mv = m_vu[nx];
      acc_t aT;   // A^T: rows j, columns k
      zero(aT);
#pragma unroll
      for (int s = 0; s < KS; ++s) mma(aT, pk.f[s], fq.f[s]);
      pk.load(ku + nx * E);
#pragma unroll
      for (int r = 0; r < 16; ++r) aT[r] = fast_rcp(__builtin_fmaf(fast_exp2(aT[r] * z), kUnitInv, kUnitInv));
      if (jt == kt) {   // j > k only
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (acc_row(r, g) <= c) aT[r] = 0.f;
      }
      const split8 fa[2] = {chain_split(aT, 0), chain_split(aT, 1)};
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        acc_t t;
        zero(t);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) mma(t, ld_free_split<HD>(s_vu, 32 * nt, 16 * s2, c, g), fa[s2]);
        add_scaled(st[nt], t, v_mul);
      }
    }
  };
  if (seg < nblk - Kb) {   // more than one part: the sums of the parts in front of this wave's
    if (hi < nblk) sweep(false);
    float* red = reinterpret_cast<float*>(castle_smem);
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
        for (int w = 0; w < kW - 1; ++w) sum = __builtin_fmaf(w < wave ? 1.f : 0.f, red[((w * NT + nt) * 16 + r) * 64 + lane], sum);
        st[nt][r] = sum;
      }
    __syncthreads();   // the memory holds tiles again
  }
  if (lo >= hi) return;
  sweep(true);
  if (hi == nblk && a.U.ptr != nullptr && k < L) {
    float* dst = head_ptr_mut<float>(a.U, b, h) + (int64_t)k * a.U.sl;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = 32 * nt + 8 * q + 4 * g;
        if (n < HD) st4<float>(dst + n, pack4<float>(st[nt], q));
      }
  }
}

// ---------------------------------------------------------------------------
// what the waves of a workgroup share (Qc', two tiles of Ku, T' rows: fragments), a tile of Vc each
template <int HD> constexpr int attn_split_tiles() { return max2((3 * split_elems<HD>() + split_elems<kNB>()) * 2 + kW * kTile<HD>, reduce_bytes<HD, kW>()); }
template <int HD> constexpr int attn_split_lds() { return attn_split_tiles<HD>() + kW * 64 * 8; }

template <int HD>
__global__ __launch_bounds__(64 * kW, 2) void attn_split_kernel(FwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>();
  const int L = a.s.L, BH = a.s.B * a.s.H, ntile = (L + 31) / 32, tiles = a.s.Lp / 32;
  int rank, bh;
  work_item_snake(BH, ntile, a.s.cus, rank, bh);
  const int it = ntile - 1 - rank;   // the last queries see the most keys
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const int i = 32 * it + c, I = it >> 1, half = it & 1;
  fp16_t* s_qc = reinterpret_cast<fp16_t*>(castle_smem);
  fp16_t* s_ku = s_qc + split_elems<HD>();
  fp16_t* s_t = s_ku + 2 * split_elems<HD>();
  fp16_t* s_v = s_t + split_elems<kNB>() + wave * kTileElems<HD>;
  float* s_stat = reinterpret_cast<float*>(castle_smem + attn_split_tiles<HD>());
  constexpr int E = split_elems<HD>();
  const fp16_t* qc = split_tiles<HD>(a.ws.qc_p, bh, tiles);   // pre-scaled by c1
  const fp16_t* kc = split_tiles<HD>(a.ws.kc_p, bh, tiles);
  const fp16_t* vc = split_tiles<HD>(a.ws.vc_p, bh, tiles);
  const fp16_t* qu = split_tiles<HD>(a.ws.qu_p, bh, tiles);
  const fp16_t* ku = split_tiles<HD>(a.ws.ku_p, bh, tiles);
  const fp16_t* tb = split_tiles<kNB>(a.ws.t_blk, bh, tiles);
  const fp16_t* snap = reinterpret_cast<const fp16_t*>(a.ws.usnap) + ((int64_t)bh * snap_rows(a.s.nblk) + usnap_off(I)) * 2 * HD;
  const float* m_kc = a.ws.op_mul + ((int64_t)kOpKc * BH + bh) * tiles;
  const float* m_vc = a.ws.op_mul + ((int64_t)kOpVc * BH + bh) * tiles;
  const float* m_qu = a.ws.op_mul + ((int64_t)kOpQu * BH + bh) * tiles;
  const float* m_ku = a.ws.op_mul + ((int64_t)kOpKu * BH + bh) * tiles + 2 * I;
  const float* u_mul = a.ws.u_mul + ((int64_t)bh * a.s.nblk + I) * tiles;
  const float q_mul = a.ws.op_mul[((int64_t)kOpQc * BH + bh) * tiles + it], t_mul = a.ws.t_mul[(int64_t)bh * a.s.nblk + I] * kUnitInv;
  const float z0[2] = {-a.s.scale * kLog2e * m_ku[0], -a.s.scale * kLog2e * m_ku[1]};

  if (wave < 3) {
    SplitRows<HD> f;
    f.load(wave == 0 ? qc + it * E : ku + (2 * I + wave - 1) * E);
    f.store_flat(s_qc + wave * E);
  } else {
    SplitRows<kNB> f;
    f.load(tb + it * split_elems<kNB>());
    f.store_flat(s_t);
  }
  __syncthreads();
  acc_t o[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(o[nt]);
  float m = -INFINITY, l = 0.f;

  SplitRows<HD> pq, pk, pv, nu;
  nu.clear();
  // what the tiles and the snapshot are to be multiplied with: a tile ahead too
  float n_q = 0.f, n_k = 0.f, n_v = 0.f, n_u = 0.f;
  auto multipliers = [&](int kt) __attribute__((always_inline)) {
    n_q = m_qu[kt];
    n_k = m_kc[kt];
    n_v = m_vc[kt];
    n_u = u_mul[kt];
  };
  if (wave <= it) {
    multipliers(wave);
    pq.load(qu + wave * E);
    pk.load(kc + wave * E);
    pv.load(vc + wave * E);
    if ((wave >> 1) < I) nu.load(snap + wave * E);
  }
  for (int kt = wave; kt <= it; kt += kW) {
    const int nx = min(kt + kW, it);   // the loads of the next tile are unconditional: the last iteration repeats one
    wave_lds_order<>();
    pv.store(s_v);
    wave_lds_order<>();
    pv.load(vc + nx * E);
    const float mq = n_q, s_mul = q_mul * n_k, o_mul = n_v * kUnitInv;
    float su_mul = q_mul * n_u;
    multipliers(nx);
    if ((kt >> 1) >= I) {   // keys of the own block: no state yet
      nu.clear();
      su_mul = 0.f;
    }
    // gates of the block's sources up to this tile: A^T[j rows, k lanes], used as the operand with k on the lanes
    split8 fa[2][2];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt) {
      if (jt <= half && 2 * I + jt >= kt) {
        acc_t aT;
        zero(aT);
#pragma unroll
        for (int s = 0; s < KS; ++s) mma(aT, of_rows<HD>(s_ku + jt * E, s), pq.f[s]);
#pragma unroll
        for (int r = 0; r < 16; ++r) aT[r] = fast_rcp(__builtin_fmaf(fast_exp2(aT[r] * (z0[jt] * mq)), kUnitInv, kUnitInv));
        if (2 * I + jt == kt) {   // j > k only
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (acc_row(r, g) <= c) aT[r] = 0.f;
        }
        fa[jt][0] = chain_split(aT, 0);
        fa[jt][1] = chain_split(aT, 1);
      } else {
        fa[jt][0] = zero_split();
        fa[jt][1] = zero_split();
      }
    }
    pq.load(qu + nx * E);
    acc_t s, su, sb;   // [k rows, i lanes]; su: by the state in front of the block, sb: by the block's sources
    zero(s);
    zero(su);
    zero(sb);
    if (half) {
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) mma(sb, fa[1][s2], of_rows<kNB>(s_t, 2 + s2));
    }
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) mma(sb, fa[0][s2], of_rows<kNB>(s_t, s2));   // (zero where j > i)
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const split8 f = of_rows<HD>(s_qc, ks);
      mma(su, nu.f[ks], f);
      mma(s, pk.f[ks], f);
    }
    pk.load(kc + nx * E);
    nu.load((nx >> 1) < I ? snap + nx * E : kc);
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float sut = __builtin_fmaf(sb[r], t_mul, su[r] * su_mul);
      const float sg = fast_rcp(1.f + fast_exp2(-sut));
      s[r] = __builtin_fmaf(-sut, sg, s[r] * s_mul);
    }
    if (kt == it) {   // causal mask
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (acc_row(r, g) > c) s[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
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
      s[r] = fast_exp2(s[r] - m);
      l += s[r];
    }
    split8 fp[2];   // (times kUnit here: 12 more in the exponent would cost it three bits)
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) fp[s2] = chain_split(s, s2, kUnit);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      acc_t t;
      zero(t);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) mma_full(t, ld_free_split<HD>(s_v, 32 * nt, 16 * s2, c, g), fp[s2]);
      add_scaled(o[nt], t, o_mul);
    }
  }
  // merge the waves: common maximum, then weighted sums
  l += __shfl_xor(l, 32);
  s_stat[(wave * 64 + lane) * 2] = m;
  s_stat[(wave * 64 + lane) * 2 + 1] = l;
  __syncthreads();
  float M = -INFINITY, lt = 0.f;
#pragma unroll
  for (int w = 0; w < kW; ++w) M = fmaxf(M, s_stat[(w * 64 + lane) * 2]);
#pragma unroll
  for (int w = 0; w < kW; ++w) {
    const float mw = s_stat[(w * 64 + lane) * 2];
    lt += mw == -INFINITY ? 0.f : fast_exp2(mw - M) * s_stat[(w * 64 + lane) * 2 + 1];
  }
  const float wt = m == -INFINITY ? 0.f : fast_exp2(m - M) / lt;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[nt][r] *= wt;
  float* dst = head_ptr_mut<float>(a.out, b, h) + (int64_t)i * a.out.sl;
  reduce_waves<kW, NT>(reinterpret_cast<float*>(castle_smem), o, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    const int n = 32 * nt + 8 * q + 4 * g;
    if (i < L && n < HD) st4<float>(dst + n, v);
  });
  if (wave == 0 && g == 0 && i < L) a.ws.lse[(int64_t)bh * a.s.Lp + i] = (M + __builtin_log2f(lt)) * kLn2;
}

// ---------------------------------------------------------------------------
// delta = rowsum(dO * O) and the copy of dO, a tile of 32 rows per wave
template <int HD>
__global__ __launch_bounds__(64 * kW) void delta_split_kernel(BwdArgs a) {
  constexpr int N = HD / 16, VPR = HD / 8;
  const int bh = blockIdx.y, b = bh / a.s.H, h = bh % a.s.H, tiles = a.s.Lp / 32, tile = blockIdx.x * kW + wave_id();
  vec<float, 8> x[N], o[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int64_t row = 32 * (int64_t)tile + lane_id() / VPR + n * (64 / VPR);
    x[n] = o[n] = zero_frag<float>();
    if (row < a.s.L) {
      x[n] = *reinterpret_cast<const frag_mem<float>*>(head_ptr<float>(a.dout, b, h) + row * a.dout.sl + lane_id() % VPR * 8);
      o[n] = *reinterpret_cast<const frag_mem<float>*>(head_ptr<float>(a.out, b, h) + row * a.out.sl + lane_id() % VPR * 8);
    }
  }
  const float inv = store_split_tile<HD>(reinterpret_cast<fp16_t*>(a.dout_p) + ((int64_t)bh * tiles + tile) * split_elems<HD>(), x);
  if (lane_id() == 0) a.do_mul[(int64_t)bh * tiles + tile] = inv;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) d = __builtin_fmaf(o[n][e], x[n][e], d);
#pragma unroll
    for (int q = 1; q < VPR; q <<= 1) d += __shfl_xor(d, q);
    if (lane_id() % VPR == 0) a.delta[(int64_t)bh * a.s.Lp + 32 * tile + (lane_id() + 64 * n) / VPR] = d;
  }
}

// ---------------------------------------------------------------------------
// shared rows of the keys (Qu, Kc, Vc); two operand tiles and the row sums of a block (-log2 normaliser, -delta) per wave
template <int HD> constexpr int key_split_wave_bytes() { return 2 * kTile<HD> + 2 * kNB * 4; }
template <int HD> constexpr int key_split_lds() { return 3 * 2 * split_elems<HD>() + max2(kW * key_split_wave_bytes<HD>(), reduce_bytes<HD, kW>()); }

template <int HD>
__global__ __launch_bounds__(64 * kW, 1) void key_split_kernel(BwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>(), KG = 2 * NT;
  const int L = a.s.L, BH = a.s.B * a.s.H, nblk = (L + kNB - 1) / kNB, tiles = a.s.Lp / 32;
  int kt, bh;   // key tile 0 meets every query
  work_item(BH, kt, bh);
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const float c0 = a.s.scale;
  const int kw0 = 32 * kt, k = kw0 + c, Iw = kt >> 1;
  fp16_t* s_qu = reinterpret_cast<fp16_t*>(castle_smem);
  fp16_t* s_kc = s_qu + split_elems<HD>();
  fp16_t* s_vc = s_kc + split_elems<HD>();
  unsigned char* work = castle_smem + 3 * 2 * split_elems<HD>();
  fp16_t* s_a = reinterpret_cast<fp16_t*>(work + wave * key_split_wave_bytes<HD>());
  fp16_t* s_b = s_a + kTileElems<HD>;
  float* s_sum = reinterpret_cast<float*>(s_b + kTileElems<HD>);
  float* red = reinterpret_cast<float*>(work);
  constexpr int E = split_elems<HD>(), ET = split_elems<kNB>();
  const fp16_t* qc = split_tiles<HD>(a.ws.qc_p, bh, tiles);
  const fp16_t* ku = split_tiles<HD>(a.ws.ku_p, bh, tiles);
  const fp16_t* vu = split_tiles<HD>(a.ws.vu_p, bh, tiles);
  const fp16_t* dout = split_tiles<HD>(a.dout_p, bh, tiles);
  const fp16_t* tb = split_tiles<kNB>(a.ws.t_blk, bh, tiles);
  const fp16_t* ttb = split_tiles<kNB>(a.ws.tt_blk, bh, tiles);
  const fp16_t* usnap = reinterpret_cast<const fp16_t*>(a.ws.usnap) + (int64_t)bh * snap_rows(a.s.nblk) * 2 * HD;
  fp16_t* gsnap = reinterpret_cast<fp16_t*>(a.gsnap) + (int64_t)bh * snap_rows(a.s.nblk) * 2 * HD;
  auto mul_of = [&](int op) __attribute__((always_inline)) { return a.ws.op_mul + ((int64_t)op * BH + bh) * tiles; };
  const float *m_qc = mul_of(kOpQc), *m_ku = mul_of(kOpKu), *m_vu = mul_of(kOpVu), *m_do = a.do_mul + (int64_t)bh * tiles;
  const float *t_mul = a.ws.t_mul + (int64_t)bh * a.s.nblk, *u_mul = a.ws.u_mul + (int64_t)bh * a.s.nblk * tiles + kt;
  const float z0 = -c0 * kLog2e * mul_of(kOpQu)[kt], k_mul = mul_of(kOpKc)[kt], v_mul = mul_of(kOpVc)[kt];
  // dS / dSu tiles of these keys, 2048 halves each: the high halves, then the low ones; of either, element (key k, chained slot) at s2 * 512 + k * 16 + g * 8
  const int64_t row0 = ((int64_t)bh * tiles + kt) * tiles;
  const uint32_t tile_at = (c * 16 + g * 8) * 2;
  fp16_t* ds_mat = reinterpret_cast<fp16_t*>(a.ds_mat) + row0 * 2048;
  fp16_t* dsu_mat = reinterpret_cast<fp16_t*>(a.dsu_mat) + row0 * 2048;
  float* ds_mul = a.ds_mul + row0;
  float* g_mul = a.g_mul + (int64_t)bh * a.s.nblk * tiles + kt;
  const float* lse = a.ws.lse + (int64_t)bh * a.s.Lp;
  const float* delta = a.delta + (int64_t)bh * a.s.Lp;

  if (wave < 3) {
    SplitRows<HD> f;
    f.load(split_tiles<HD>(wave == 0 ? a.ws.qu_p : wave == 1 ? a.ws.kc_p : a.ws.vc_p, bh, tiles) + kt * E);
    f.store_flat(s_qu + wave * E);
  }
  const int seg = (nblk - Iw + kW - 1) / kW;
  const int lo = min(nblk, Iw + wave * seg), hi = min(nblk, lo + seg);
  // gate A^T[j rows, k lanes] of source tile jt from its Ku rows, times 1 / `one`
  auto gate = [&](acc_t& aT, const SplitRows<HD>& rows, int jt, float one) __attribute__((always_inline)) {
    const float z = z0 * m_ku[jt];
    zero(aT);
#pragma unroll
    for (int s = 0; s < KS; ++s) mma(aT, rows.f[s], of_rows<HD>(s_qu, s));
#pragma unroll
    for (int r = 0; r < 16; ++r) aT[r] = fast_rcp(__builtin_fmaf(fast_exp2(aT[r] * z), one, one));
    if (jt <= kt) {   // j > k only
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * (jt - kt) + acc_row(r, g) <= c) aT[r] = 0.f;
    }
  };
  // the next tiles, requested one step ahead
  SplitRows<HD> pa, pb;
  SplitRows<kNB> pt;

  acc_t G[NT];   // [n rows, k lanes]
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(G[nt]);
  {
    // ---- pass A: score chain, dVc, dKc, this part's contribution to the reverse state -------------------------------
    acc_t dvc[NT], dkc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) { zero(dvc[nt]); zero(dkc[nt]); }
    float nl = 0.f, nd = 0.f;   // one row of the block per lane, a block ahead
    auto sums = [&](int I) __attribute__((always_inline)) {
      nl = load_at<float>(lse + I * kNB, 4 * lane);
      nd = load_at<float>(delta + I * kNB, 4 * lane);
    };
    if (lo < hi) {
      pa.load(ku + 2 * lo * E);
      pb.load(ku + (2 * lo + 1) * E);
      sums(lo);
    }
    __syncthreads();   // the shared rows are there
    for (int I = lo; I < hi; ++I) {
      const bool there = I * kNB + lane < L;
      s_sum[lane] = there ? -nl * kLog2e : -INFINITY;
      s_sum[kNB + lane] = there ? -nd : 0.f;
      sums(min(I + 1, nblk - 1));
      SplitRows<HD> fub;
      fub.load(I > Iw ? usnap + (usnap_off(I) + kw0) * 2 * HD : ku);
      const float su0 = I > Iw ? u_mul[(int64_t)I * tiles] : 0.f, tm = t_mul[I] * kUnitInv;
      split8 fa[2][2];
      {
        acc_t a0, a1;
        gate(a0, pa, 2 * I, kUnitInv);
        pa.load(qc + 2 * I * E);
        gate(a1, pb, 2 * I + 1, kUnitInv);
        pb.load(dout + 2 * I * E);
        pt.load(tb + 2 * I * ET);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) { fa[0][s2] = chain_split(a0, s2); fa[1][s2] = chain_split(a1, s2); }
      }
      if (I == Iw) fub.clear();   // no state in front of the keys' own block
#pragma unroll
      for (int itl = 0; itl < 2; ++itl) {
        const int it = 2 * I + itl;
        acc_t p, su, sb, dp;   // [i rows, k lanes]; su: by the state in front of the block, sb: by the block's sources
        zero(p);
        zero(su);
        zero(sb);
        zero(dp);
        wave_lds_order<>();
        pa.store(s_a);
        pb.store(s_b);
        wave_lds_order<>();
        if (itl == 0) {
          pa.load(qc + (2 * I + 1) * E);
          pb.load(dout + (2 * I + 1) * E);
        } else {
          const int nx = min(I + 1, nblk - 1);
          pa.load(ku + 2 * nx * E);
          pb.load(ku + (2 * nx + 1) * E);
        }
        const float qm = m_qc[it], dm = m_do[it];
        const float s_mul = qm * k_mul, su_mul = qm * su0, dp_mul = dm * v_mul;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const split8 oq = ld_nat_split<HD>(s_a, c, 16 * s + 8 * g);
          mma(su, oq, fub.f[s]);
          mma(p, oq, of_rows<HD>(s_kc, s));
          mma(dp, ld_nat_split<HD>(s_b, c, 16 * s + 8 * g), of_rows<HD>(s_vc, s));
        }
#pragma unroll
        for (int jt = 0; jt < 2; ++jt)
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2)
            if (jt <= itl) mma(sb, pt.f[2 * jt + s2], fa[jt][s2]);
        if (itl == 0) pt.load(tb + (2 * I + 1) * ET);
        acc_t ds, dsu;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const vec<float, 4> l4 = *reinterpret_cast<const vec<float, 4>*>(s_sum + 32 * itl + 8 * q + 4 * g);
          const vec<float, 4> d4 = *reinterpret_cast<const vec<float, 4>*>(s_sum + kNB + 32 * itl + 8 * q + 4 * g);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int r = 4 * q + e;
            const float lr = it <= kt && 32 * (it - kt) + acc_row(r, g) < c ? -INFINITY : l4[e];   // queries before the key see nothing
            const float sut = __builtin_fmaf(sb[r], tm, su[r] * su_mul);  // log2(e) * Su
            const float sg = fast_rcp(1.f + fast_exp2(-sut));
            const float w = fast_exp2(__builtin_fmaf(-sut, sg, __builtin_fmaf(p[r], s_mul, lr)));
            const float dsv = w * __builtin_fmaf(dp[r], dp_mul, d4[e]);
            const float y = sut * kLn2;                                   // true Su
            const float t = __builtin_fmaf(-y, sg, y);                    // y (1 - sigmoid)
            const float sp = __builtin_fmaf(sg, t, sg);                   // silu'(y), at most 1.1
            p[r] = w;
            ds[r] = dsv;
            dsu[r] = -dsv * sp;
          }
        }
        const TileScale ts = tile_scale(wave_max_bits(abs_max(ds)));
        if (lane == 0) ds_mul[it] = ts.inv;
        const float q_mul = ts.inv * qm, d_mul = dm * kUnitInv;
        split8 fp[2], fds[2], fdsu[2];
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) {
          fp[s2] = chain_split(p, s2, kUnit);
          fds[s2] = chain_split(ds, s2, ts.mul);
          fdsu[s2] = chain_split(dsu, s2, ts.mul);
          fp16_t* dst = ds_mat + (int64_t)it * 2048 + s2 * 512;
          store_at<frag_mem<fp16_t>>(dst, tile_at, fds[s2].h);   // whole lines per store
          store_at<frag_mem<fp16_t>>(dst + 1024, tile_at, fds[s2].l);
          dst = dsu_mat + (int64_t)it * 2048 + s2 * 512;
          store_at<frag_mem<fp16_t>>(dst, tile_at, fdsu[s2].h);
          store_at<frag_mem<fp16_t>>(dst + 1024, tile_at, fdsu[s2].l);
        }
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          acc_t t1, t2, t3;
          zero(t1);
          zero(t2);
          zero(t3);
#pragma unroll
          for (int s2 = 0; s2 < 2; ++s2) {
            const split8 qt = ld_free_split<HD>(s_a, 32 * nt, 16 * s2, c, g);
            mma(t1, qt, fds[s2]);
            mma(t2, qt, fdsu[s2]);
            mma(t3, ld_free_split<HD>(s_b, 32 * nt, 16 * s2, c, g), fp[s2]);
          }
          add_scaled(dvc[nt], t3, d_mul);
          add_scaled(dkc[nt], t1, q_mul);
          add_scaled(G[nt], t2, q_mul);
        }
      }
    }
    float* row = head_ptr_mut<float>(a.dkc, b, h) + (int64_t)k * a.dkc.sl;
    reduce_waves<kW, NT>(red, dkc, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
      if (k < L) store_quad<float, HD>(row, 32 * nt + 8 * q + 4 * g, v, kLn2, a.s.rotary ? k : -1);
    });
    row = head_ptr_mut<float>(a.dvc, b, h) + (int64_t)k * a.dvc.sl;
    reduce_waves<kW, NT>(red, dvc, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
      if (k < L) store_quad<float, HD>(row, 32 * nt + 8 * q + 4 * g, v, 1.f, -1);
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
      for (int w = 1; w < kW; ++w) sum = __builtin_fmaf(w > wave ? 1.f : 0.f, red[((w * NT + nt) * 16 + r) * 64 + lane], sum);
      G[nt][r] = sum;
    }
  __syncthreads();   // the memory holds tiles again
  // ---- pass B: from the last block of the part down ------------------------------------------------------------------
  acc_t dqu[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) zero(dqu[nt]);
  auto request = [&](int I, int jtl) __attribute__((always_inline)) {   // the source tile 2 I + jtl
    pa.load(ku + (2 * I + jtl) * E);
    pb.load(vu + (2 * I + jtl) * E);
    pt.load(ttb + (2 * I + jtl) * ET);
  };
  // (this wave stored them in pass A: through the vector cache, a block ahead)
  auto mul_of_block = [&](int I) __attribute__((always_inline)) { return load_at<vec<float, 2>>(ds_mul + 2 * I, 0); };
  vec<float, 2> f_next = {0.f, 0.f};
  if (lo < hi) {
    request(hi - 1, 0);
    f_next = mul_of_block(hi - 1);
  }
  for (int I = hi - 1; I >= lo; --I) {
    split8 fdsu[2][2];   // this wave stored them in pass A
    const float f_mul[2] = {f_next[0], f_next[1]};
    f_next = mul_of_block(max(I - 1, lo));
#pragma unroll
    for (int itl = 0; itl < 2; ++itl) {
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const fp16_t* src = dsu_mat + (int64_t)(2 * I + itl) * 2048 + s2 * 512;
        fdsu[itl][s2] = split8{load_at<frag_mem<fp16_t>>(src, tile_at), load_at<frag_mem<fp16_t>>(src + 1024, tile_at)};
      }
    }
    settle();
    float gm = abs_max(G[0]);
#pragma unroll
    for (int nt = 1; nt < NT; ++nt) gm = abs_max(G[nt], gm);
    const TileScale gs = tile_scale(wave_max_bits(gm));
    split8 fg[KG];
#pragma unroll
    for (int s = 0; s < KG; ++s) fg[s] = chain_split(G[s / 2], s % 2, gs.mul);
    if (I <= nblk - 2) {
      store_snap_halves<HD>(gsnap + (gsnap_off(I) + kw0) * 2 * HD, fg, c, g);
      if (lane == 0) g_mul[(int64_t)I * tiles] = gs.inv;
    }
#pragma unroll
    for (int jtl = 0; jtl < 2; ++jtl) {
      wave_lds_order<>();
      pa.store(s_a);
      wave_lds_order<>();
      const float a_mul = m_vu[2 * I + jtl] * gs.inv;
      acc_t aT, dA, t;   // [j rows, k lanes]
      gate(aT, pa, 2 * I + jtl, 1.f);
      pa.load(jtl == 0 ? ku + (2 * I + 1) * E : qc + 2 * I * E);
      zero(t);
#pragma unroll
      for (int s = 0; s < KS; ++s) mma(t, chained(pb.f[s]), fg[s]);
      pb.load(jtl == 0 ? vu + (2 * I + 1) * E : qc + (2 * I + 1) * E);
#pragma unroll
      for (int r = 0; r < 16; ++r) dA[r] = t[r] * a_mul;
#pragma unroll
      for (int itl = 0; itl < 2; ++itl) {
        if (itl < jtl) continue;
        zero(t);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) mma(t, pt.f[2 * itl + s2], fdsu[itl][s2]);
        add_scaled(dA, t, t_mul[I] * f_mul[itl]);
      }
      if (jtl == 0) pt.load(ttb + (2 * I + 1) * ET);
#pragma unroll
      for (int r = 0; r < 16; ++r) dA[r] *= __builtin_fmaf(-aT[r], aT[r], aT[r]);   // dZ = dA A (1 - A)
      const TileScale zs = tile_scale(wave_max_bits(abs_max(dA)));
      split8 fdz[2];
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) fdz[s2] = chain_split(dA, s2, zs.mul);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        zero(t);
#pragma unroll
        for (int s2 = 0; s2 < 2; ++s2) mma(t, ld_free_split<HD>(s_a, 32 * nt, 16 * s2, c, g), fdz[s2]);
        add_scaled(dqu[nt], t, m_ku[2 * I + jtl] * zs.inv);
      }
    }
    // the block joins the reverse state
    wave_lds_order<>();
    pa.store(s_a);
    pb.store(s_b);
    wave_lds_order<>();
    request(max(I - 1, 0), 0);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      acc_t t0, t1;
      zero(t0);
      zero(t1);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        mma(t0, ld_free_split<HD>(s_a, 32 * nt, 16 * s2, c, g), fdsu[0][s2]);
        mma(t1, ld_free_split<HD>(s_b, 32 * nt, 16 * s2, c, g), fdsu[1][s2]);
      }
      add_scaled(G[nt], t0, m_qc[2 * I] * f_mul[0]);
      add_scaled(G[nt], t1, m_qc[2 * I + 1] * f_mul[1]);
    }
  }
  float* row = head_ptr_mut<float>(a.dqu, b, h) + (int64_t)k * a.dqu.sl;
  reduce_waves<kW, NT>(red, dqu, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    if (k < L) store_quad<float, HD>(row, 32 * nt + 8 * q + 4 * g, v, c0 * kLn2, a.s.rotary ? k : -1);
  });
}

// ---------------------------------------------------------------------------
template <int HD> constexpr int query_split_wave_bytes() { return 2 * kTile<HD> + 2 * split_tile_bytes<32>(); }
template <int HD> constexpr int query_split_lds() { return 3 * kTile<HD> + 2 * split_elems<kNB>() + max2(kW * query_split_wave_bytes<HD>(), reduce_bytes<HD, kW>()); }

template <int HD>
__global__ __launch_bounds__(64 * kW, 1) void query_split_kernel(BwdArgs a) {
  constexpr int KS = HD / 16, NT = narrow_nt<HD>();
  const int L = a.s.L, BH = a.s.B * a.s.H, ntile = (L + 31) / 32, nblk = (L + kNB - 1) / kNB, tiles = a.s.Lp / 32;
  int rank, bh;
  work_item(BH, rank, bh);
  const int it = ntile - 1 - rank;   // the last rows meet the most keys
  const int b = bh / a.s.H, h = bh % a.s.H;
  const int lane = lane_id(), wave = wave_id(), c = lane & 31, g = lane >> 5;
  const float c0 = a.s.scale;
  const int i = 32 * it + c, I = it >> 1, half = it & 1;
  const bool has_g = I <= nblk - 2;                     // a reverse state exists behind the block
  const bool next = half == 0 && it + 1 < ntile;        // the block's second tile of queries exists and is not this one
  // the rows of the tile as sources (Ku, Vu) and, for a second tile, the Ku rows of the block's first one, whose sources its queries meet
  // too; shared by the waves
  fp16_t* s_ku = reinterpret_cast<fp16_t*>(castle_smem);
  fp16_t* s_vu = s_ku + kTileElems<HD>;
  fp16_t* s_k0 = s_vu + kTileElems<HD>;
  fp16_t* s_tt = s_k0 + kTileElems<HD>;   // T'^T rows of the tile: fragments
  unsigned char* work = castle_smem + 3 * kTile<HD> + 2 * split_elems<kNB>();
  fp16_t* s_x = reinterpret_cast<fp16_t*>(work + wave * query_split_wave_bytes<HD>());
  fp16_t* s_y = s_x + kTileElems<HD>;
  fp16_t* s_ds = s_y + kTileElems<HD>;
  fp16_t* s_dsu = s_ds + kTileElems<32>;
  float* red = reinterpret_cast<float*>(work);
  constexpr int E = split_elems<HD>();
  const fp16_t* qc = split_tiles<HD>(a.ws.qc_p, bh, tiles);
  const fp16_t* kc = split_tiles<HD>(a.ws.kc_p, bh, tiles);
  const fp16_t* qu = split_tiles<HD>(a.ws.qu_p, bh, tiles);
  const fp16_t* ku = split_tiles<HD>(a.ws.ku_p, bh, tiles);
  const fp16_t* vu = split_tiles<HD>(a.ws.vu_p, bh, tiles);
  const fp16_t* ttb = split_tiles<kNB>(a.ws.tt_blk, bh, tiles);
  const fp16_t* usnap = reinterpret_cast<const fp16_t*>(a.ws.usnap) + ((int64_t)bh * snap_rows(a.s.nblk) + usnap_off(I)) * 2 * HD;
  const fp16_t* gsnap = reinterpret_cast<const fp16_t*>(a.gsnap) + ((int64_t)bh * snap_rows(a.s.nblk) + (has_g ? gsnap_off(I) : 0)) * 2 * HD;
  const int64_t row0 = (int64_t)bh * tiles * tiles + it;   // + kt * tiles
  const fp16_t* ds_mat = reinterpret_cast<const fp16_t*>(a.ds_mat);
  const fp16_t* dsu_mat = reinterpret_cast<const fp16_t*>(a.dsu_mat);
  const float* g_mul = a.g_mul + ((int64_t)bh * a.s.nblk + I) * tiles;
  const uint32_t tile_at = (c * 16 + g * 8) * 2;
  auto mul_of = [&](int op) __attribute__((always_inline)) { return a.ws.op_mul + ((int64_t)op * BH + bh) * tiles; };
  const float *m_kc = mul_of(kOpKc), *m_qu = mul_of(kOpQu), *m_qc = mul_of(kOpQc), *m_vu = mul_of(kOpVu), *u_mul = a.ws.u_mul + ((int64_t)bh * a.s.nblk + I) * tiles;
  const float zK = -c0 * kLog2e * mul_of(kOpKu)[it], z0 = -c0 * kLog2e * mul_of(kOpKu)[2 * I], v_mul = m_vu[it], t_mul = a.ws.t_mul[(int64_t)bh * a.s.nblk + I];

  if (wave < 3) {
    SplitRows<HD> f;
    f.load(wave == 0 ? ku + it * E : wave == 1 ? vu + it * E : ku + 2 * I * E);
    f.store(s_ku + wave * kTileElems<HD>);
  } else {
    SplitRows<kNB> f;
    f.load(ttb + it * split_elems<kNB>());
    f.store_flat(s_tt);
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

  auto load_tile = [&](split8 (&f)[2], const fp16_t* tile) __attribute__((always_inline)) {
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) f[s2] = split8{load_at<frag_mem<fp16_t>>(tile + s2 * 512, tile_at), load_at<frag_mem<fp16_t>>(tile + 1024 + s2 * 512, tile_at)};
  };
  // a tile in natural query order, [key][query], to be read with the query on the lanes
  auto put_tile = [&](fp16_t* tile, const split8 (&f)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const frag<fp16_t>& x = p == 0 ? f[s2].h : f[s2].l;
        vec<fp16_t, 4> lo, hi;
#pragma unroll
        for (int e = 0; e < 4; ++e) { lo[e] = x[e]; hi[e] = x[4 + e]; }
        fp16_t* dst = tile + p * split_plane<32>() + c * split_ld<32>() + 16 * s2 + 4 * g;
        st4<fp16_t>(dst, lo);
        st4<fp16_t>(dst + 8, hi);
      }
  };
  SplitRows<HD> pq;   // a key tile ahead
  pq.load(qu + min(wave, it) * E);
  for (int kt = wave; kt <= it; kt += kW) {
    const int Kb = kt >> 1;
    const int64_t row = row0 + (int64_t)kt * tiles;
    SplitRows<HD> pk, ou, og;
    split8 fds[2], fdsu[2], fdsn[2];
    load_tile(fdsu, dsu_mat + row * 2048);
    load_tile(fdsn, dsu_mat + (row + (next ? 1 : 0)) * 2048);
    og.load(has_g ? gsnap + kt * E : kc);
    const float f_it = a.ds_mul[row], f_nx = a.ds_mul[row + (next ? 1 : 0)], f_g = has_g ? g_mul[kt] : 0.f, mq = m_qu[kt], f_k = m_kc[kt];
    const float f_u = Kb < I ? u_mul[kt] : 0.f;
    wave_lds_order<>();
    pq.store(s_x);
    // gates A[k rows, j lanes] of the own sources, and of the first tile's sources for a second tile (zero where they do
    // not lie behind the keys), times kUnit
    acc_t aK, a0;
    zero(aK);
    zero(a0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      mma(a0, pq.f[s], ld_nat_split<HD>(s_k0, c, 16 * s + 8 * g));
      mma(aK, pq.f[s], ld_nat_split<HD>(s_ku, c, 16 * s + 8 * g));
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      aK[r] = fast_rcp(__builtin_fmaf(fast_exp2(aK[r] * (zK * mq)), kUnitInv, kUnitInv));
      a0[r] = fast_rcp(__builtin_fmaf(fast_exp2(a0[r] * (z0 * mq)), kUnitInv, kUnitInv));
    }
    if (kt + 1 >= it) {   // j > k only
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (c + 32 * (it - kt) <= acc_row(r, g)) aK[r] = 0.f;
        if (c + 32 * (2 * I - kt) <= acc_row(r, g)) a0[r] = 0.f;
      }
    }
    split8 fa[2], f0[2];
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) { fa[s2] = chain_split(aK, s2); f0[s2] = chain_split(a0, s2); }
    if (!next) {
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) fdsn[s2] = zero_split();
    }
    if (!has_g) og.clear();
    put_tile(s_dsu, fdsu);
    put_tile(s_ds, fdsn);
    og.store(s_y);
    wave_lds_order<>();
    load_tile(fds, ds_mat + row * 2048);
    split8 bdsu[2];
    acc_t t1, t2;
    zero(t1);
    zero(t2);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      bdsu[s2] = ld_free_split<32>(s_dsu, 0, 16 * s2, c, g);
      const split8 bdsn = ld_free_split<32>(s_ds, 0, 16 * s2, c, g);
      mma(t1, fa[s2], bdsu[s2]);
      // one of the two products, chosen by operands: the second tile of the block, or the first (zeros without a second)
      mma(t2, half == 1 ? f0[s2] : bdsn, half == 1 ? bdsu[s2] : fa[s2]);
    }
    add_scaled(own, t1, f_it * kUnitInv);
    add_scaled(far, t2, (half == 1 ? f_it : f_nx) * kUnitInv);
    wave_lds_order<>();
    put_tile(s_ds, fds);
    pk.load(kc + kt * E);
    ou.load(Kb < I ? usnap + kt * E : kc);
    // dA = dSu^T T' + G' Vu^T, dZ, dKu, dVu
    acc_t dA;
    zero(dA);
    zero(t1);
    zero(t2);
#pragma unroll
    for (int s = 0; s < KS; ++s) mma(dA, og.f[s], ld_nat_split<HD>(s_vu, c, 16 * s + 8 * g));
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      mma(t1, fdsu[s2], of_rows<kNB>(s_tt, 2 * half + s2));
      mma(t2, fdsn[s2], of_rows<kNB>(s_tt, 2 + s2));   // (zeros without a next tile)
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float d = __builtin_fmaf(dA[r], f_g * v_mul, __builtin_fmaf(t1[r], f_it * t_mul, t2[r] * (f_nx * t_mul)));
      dA[r] = d * (aK[r] * __builtin_fmaf(aK[r], -kUnitInv * kUnitInv, kUnitInv));   // A (1 - A) from A times kUnit
    }
    const TileScale zs = tile_scale(wave_max_bits(abs_max(dA)));
    split8 fdz[2];
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) fdz[s2] = chain_split(dA, s2, zs.mul);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      zero(t1);
      zero(t2);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        mma(t1, ld_free_split<HD>(s_x, 32 * nt, 16 * s2, c, g), fdz[s2]);
        mma(t2, ld_free_split<HD>(s_y, 32 * nt, 16 * s2, c, g), fa[s2]);
      }
      add_scaled(dku[nt], t1, zs.inv * mq);
      add_scaled(dvu[nt], t2, f_g * kUnitInv);
    }
    wave_lds_order<>();
    pq.load(qu + min(kt + kW, it) * E);   // (unconditional: the last iteration repeats a tile)
    if (Kb >= I) ou.clear();
    pk.store(s_x);
    ou.store(s_y);
    wave_lds_order<>();
    split8 bds[2];
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) bds[s2] = ld_free_split<32>(s_ds, 0, 16 * s2, c, g);
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      zero(t1);
      zero(t2);
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        mma(t1, ld_free_split<HD>(s_x, 32 * nt, 16 * s2, c, g), bds[s2]);
        mma(t2, ld_free_split<HD>(s_y, 32 * nt, 16 * s2, c, g), bdsu[s2]);
      }
      add_scaled(dqc[nt], t1, f_it * f_k);
      add_scaled(dqc[nt], t2, f_it * f_u);
    }
  }
  // ---- epilogue: dT inside the block:  dqc += dT Vu,  dvu += dT^T Qc' ---------------------------------------------------
  total_of_waves<kW>(red, own, wave, lane);
  total_of_waves<kW>(red, far, wave, lane);
  __syncthreads();   // the memory holds tiles again
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if (acc_row(r, g) > c) own[r] = 0.f;   // j <= i
  const TileScale os = tile_scale(wave_max_bits(abs_max(own))), fs = tile_scale(wave_max_bits(abs_max(far)));
  split8 fo[2], ff[2];
#pragma unroll
  for (int s2 = 0; s2 < 2; ++s2) { fo[s2] = chain_split(own, s2, os.mul); ff[s2] = chain_split(far, s2, fs.mul); }
  put_tile(s_ds, fo);   // the own tile with i as the contraction: X[i][j]
  // the Qc' rows of the tile; a second tile: the first tile's Vu rows (for dqc), a first tile: the second tile's Qc' rows
  SplitRows<HD> pi, pk;
  const int nx = min(it + 1, tiles - 1);
  pi.load(qc + it * E);
  pk.load(half == 1 ? vu + 2 * I * E : qc + nx * E);
  pi.store(s_y);
  pk.store(s_x);
  wave_lds_order<>();
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    if (nt % kW != wave) continue;   // every column tile once
    acc_t t0, t1, t2;
    zero(t0);
    zero(t1);
    zero(t2);
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      mma(t0, ld_free_split<HD>(s_x, 32 * nt, 16 * s2, c, g), ff[s2]);
      mma(t1, ld_free_split<HD>(s_vu, 32 * nt, 16 * s2, c, g), fo[s2]);
      mma(t2, ld_free_split<HD>(s_y, 32 * nt, 16 * s2, c, g), ld_free_split<32>(s_ds, 0, 16 * s2, c, g));
    }
    add_scaled(dqc[nt], t1, os.inv * v_mul);
    add_scaled(dvu[nt], t2, os.inv * m_qc[it]);
    const float f_mul = fs.inv * (half == 1 ? m_vu[2 * I] : m_qc[nx]);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float x = t0[r] * f_mul;
      dqc[nt][r] += half == 1 ? x : 0.f;
      dvu[nt][r] += half == 1 ? 0.f : x;
    }
  }
  const int pos = a.s.rotary ? i : -1;
  float* row = head_ptr_mut<float>(a.dqc, b, h) + (int64_t)i * a.dqc.sl;
  reduce_waves<kW, NT>(red, dqc, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    if (i < L) store_quad<float, HD>(row, 32 * nt + 8 * q + 4 * g, v, c0, pos);
  });
  row = head_ptr_mut<float>(a.dku, b, h) + (int64_t)i * a.dku.sl;
  reduce_waves<kW, NT>(red, dku, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    if (i < L) store_quad<float, HD>(row, 32 * nt + 8 * q + 4 * g, v, c0 * kLn2, pos);
  });
  row = head_ptr_mut<float>(a.dvu, b, h) + (int64_t)i * a.dvu.sl;
  reduce_waves<kW, NT>(red, dvu, wave, lane, [&](int nt, int q, vec<float, 4> v) __attribute__((always_inline)) {
    if (i < L) store_quad<float, HD>(row, 32 * nt + 8 * q + 4 * g, v, kLn2, pos);
  });
}

// ---------------------------------------------------------------------------
template <typename K> static bool raise_lds(K kernel, int bytes) {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes) == hipSuccess;
}

int launch_prep_split(const FwdArgs& a, hipStream_t stream) {
  return by_head_dim<float>(a.s.d, [&](auto hd) {
    constexpr int HD = decltype(hd)::value;
    ProfScope ps(kSlotPrep, stream);
    hipLaunchKernelGGL((prep_split_kernel<HD>), dim3(a.s.Lp / 32 / kW, a.s.B * a.s.H, 6), dim3(64 * kW), 0, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -3;
  });
}
int launch_scan_split(const FwdArgs& a, hipStream_t stream) {
  return by_head_dim<float>(a.s.d, [&](auto hd) {
    constexpr int HD = decltype(hd)::value, lds = scan_split_lds<HD>();
    static_assert(2 * lds <= kMaxLds);
    static PerDeviceOnce once;
    bool& configured = once.flag();
    if (!configured) configured = raise_lds(&scan_split_kernel<HD>, lds);
    if (!configured) return -3;
    const int BH = a.s.B * a.s.H, tiles = a.s.Lp / 32;
    ProfScope ps(kSlotScan, stream);
    hipLaunchKernelGGL((scan_split_kernel<HD>), dim3(tiles * BH + (a.with_t ? a.s.nblk * BH : 0)), dim3(64 * kW), lds, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -3;
  });
}
int launch_attn_split(const FwdArgs& a, hipStream_t stream) {
  return by_head_dim<float>(a.s.d, [&](auto hd) {
    constexpr int HD = decltype(hd)::value, lds = attn_split_lds<HD>();
    static_assert(lds <= kMaxLds);
    static PerDeviceOnce once;
    bool& configured = once.flag();
    if (!configured) configured = raise_lds(&attn_split_kernel<HD>, lds);
    if (!configured) return -3;
    ProfScope ps(kSlotAttn, stream);
    hipLaunchKernelGGL((attn_split_kernel<HD>), dim3((a.s.L + 31) / 32 * a.s.B * a.s.H), dim3(64 * kW), lds, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -3;
  });
}
int launch_bwd_split(const BwdArgs& a, hipStream_t stream) {
  return by_head_dim<float>(a.s.d, [&](auto hd) {
    constexpr int HD = decltype(hd)::value, key_lds = key_split_lds<HD>(), query_lds = query_split_lds<HD>();
    static_assert(key_lds <= kMaxLds && query_lds <= kMaxLds);
    static PerDeviceOnce once;
    bool& configured = once.flag();
    if (!configured) configured = raise_lds(&key_split_kernel<HD>, key_lds) && raise_lds(&query_split_kernel<HD>, query_lds);
    if (!configured) return -3;
    const dim3 grid((a.s.L + 31) / 32 * a.s.B * a.s.H);
    {
      ProfScope ps(kSlotDelta, stream);
      hipLaunchKernelGGL((delta_split_kernel<HD>), dim3(a.s.Lp / 32 / kW, a.s.B * a.s.H), dim3(64 * kW), 0, stream, a);
    }
    {
      ProfScope ps(kSlotBwdKey, stream);
      hipLaunchKernelGGL((key_split_kernel<HD>), grid, dim3(64 * kW), key_lds, stream, a);
    }
    {
      ProfScope ps(kSlotBwdQuery, stream);
      hipLaunchKernelGGL((query_split_kernel<HD>), grid, dim3(64 * kW), query_lds, stream, a);
    }
    return hipGetLastError() == hipSuccess ? 0 : -3;
  });
}

}  // namespace castle
