// CASTLE cached decode step for gfx950: one streaming pass over the cache.
//
// Reference semantics: lookahead_keys_attention.py:166-203.  For every cached row k < t
//     a_k  = sigmoid(s qu_k . ku_t)            U_k <- U_k + a_k vu_t      (in place)
//     x_k  = s qc_t . kc_k - silu(s qc_t . U_k)
// and for the appended row t:  U_t = 0,  x_t = s qc_t . kc_t;  out = softmax(x) V.
// The pass is bandwidth bound: each cached element of qu, U, kc, vc is read once and U is
// written once (5 * t * d elements per head and step).  The t rows of one (b, h) are split
// over `splits` workgroups that each keep an online-softmax partial (acc, m, l) in fp32; the last
// of them also takes row t and appends the new rows.  The partials are merged by the split that finishes last, where
// a launch in front has cleared the arrival counts (castle_decode_layer), else by decode_finish_kernel.  (Letting
// every workgroup of the output projection merge them while it loads its operand is slower: 14.7 against 13.4 us
// for a whole layer step of one sequence, 31 against 23 us for 16.)
#include "castle_tiles.h"
#include "castle_dispatch.h"
#include "castle_params.h"
#include "castle_profile.h"
#include <algorithm>
#include <mutex>
#include <type_traits>

namespace castle {

template <typename T> __device__ __forceinline__ T* view_row(const View4& v, int b, int h, int64_t row) {
  return reinterpret_cast<T*>(v.ptr) + (int64_t)b * v.sb + (int64_t)h * v.sh + row * v.sl;
}

template <typename T, int N> __device__ __forceinline__ void load_f32(const T* p, float (&dst)[N]) {
  typedef vec<T, N> vt;
  vt x = *reinterpret_cast<const vt*>(p);
#pragma unroll
  for (int e = 0; e < N; ++e) dst[e] = (float)x[e];
}

// One 16-byte piece of a U row to fp32 and back.  UH: the buffer is in the half-precision cache
// format (fp16 bits of U * kUHalfScale, saturated) whatever the element type T of the cache is.
template <typename T, int N, bool UH> __device__ __forceinline__ void u_unpack(vec<T, N> raw, float (&dst)[N]) {
  if constexpr (UH) {
    static_assert(sizeof(T) == 2, "the half-precision format replaces a 16-bit element type");
    const vec<fp16_t, N> x = __builtin_bit_cast(vec<fp16_t, N>, raw);
#pragma unroll
    for (int e = 0; e < N; ++e) dst[e] = (float)x[e] * kUHalfUnscale;
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) dst[e] = (float)raw[e];
  }
}
template <typename T, int N, bool UH> __device__ __forceinline__ vec<T, N> u_pack(const float (&src)[N]) {
  if constexpr (UH) {
    vec<fp16_t, N> x;
#pragma unroll
    for (int e = 0; e < N; ++e) x[e] = (fp16_t)__builtin_amdgcn_fmed3f(src[e] * kUHalfScale, -kHalfMax, kHalfMax);
    return __builtin_bit_cast(vec<T, N>, x);
  } else {
    vec<T, N> x;
#pragma unroll
    for (int e = 0; e < N; ++e) x[e] = (T)src[e];
    return x;
  }
}

// Sum over a group of LPR neighbouring lanes, in every lane.  The first steps move data inside the vector unit
// (DPP: neighbours, halves of eight, rows of 16); a shuffle through the LDS crossbar takes several times as long,
// and nine of them in a row per cached row are what a short step used to wait for.
template <int CTRL> __device__ __forceinline__ float dpp_add(float v) {
  const int x = __builtin_bit_cast(int, v);
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, true));
}
template <int LPR> __device__ __forceinline__ float group_sum(float v) {
  if constexpr (LPR >= 2) v = dpp_add<0xB1>(v);    // quad_perm [1, 0, 3, 2]
  if constexpr (LPR >= 4) v = dpp_add<0x4E>(v);    // quad_perm [2, 3, 0, 1]
  if constexpr (LPR >= 8) v = dpp_add<0x141>(v);   // row_half_mirror: lane i <- 7 - i of its eight
  if constexpr (LPR >= 16) v = dpp_add<0x140>(v);  // row_mirror: lane i <- 15 - i of its sixteen
  if constexpr (LPR >= 32) v += __shfl_xor(v, 16);
  return v;
}

// Folds a value over the lanes that sit at the same place of the wave's groups of LPR lanes, in every lane, inside the vector unit
// too: rotations of a row of 16, then exchanges of rows and of halves.  (Shuffles through LDS, 30 of them, took 0.3 us.)
template <int LPR, typename Op> __device__ __forceinline__ float fold_groups(float v, Op&& op) {
  auto turned = [&](auto ctrl) __attribute__((always_inline)) {
    const int x = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(x, x, decltype(ctrl)::value, 0xf, 0xf, true));
  };
  if constexpr (LPR <= 2) v = op(v, turned(std::integral_constant<int, 0x122>()));   // row_ror:2
  if constexpr (LPR <= 4) v = op(v, turned(std::integral_constant<int, 0x124>()));   // row_ror:4
  if constexpr (LPR <= 8) v = op(v, turned(std::integral_constant<int, 0x128>()));   // row_ror:8
  if constexpr (LPR <= 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    v = op(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
  }
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
  return op(__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1]));
}

// partial results of the split pass: the sums of all (b, h, split), then their statistics (maximum, sum of weights)
__device__ __forceinline__ float* part_acc(const DecodeArgs& a, int bh, int split, int HD) {
  return a.part + ((int64_t)bh * a.splits + split) * HD;
}
__device__ __forceinline__ float* part_stat(const DecodeArgs& a, int bh, int split, int HD) {
  return a.part + (int64_t)a.B * a.H * a.splits * HD + ((int64_t)bh * a.splits + split) * 2;
}

// Partials cross from one XCD's L2 to another's inside a launch: stored and loaded at agent scope (write-through, no hit in a
// stale L2), with the stores complete before the arrival is counted.  A fence would write the whole L2 back instead, dirty
// lookahead-key rows included.
__device__ __forceinline__ void agent_store(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float agent_load(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Results that cross from one job of a launch to another without a wait for the memory in between: 8-byte words of four
// payload bytes and the tag of the launch, stored and loaded at agent scope.  A word that carries the tag is there, whole.
struct TokenWords {
  const uint64_t* proj = nullptr;   // [B][6][H][d] in words
  uint64_t* merged = nullptr;       // [B][H][d]
  uint64_t* part = nullptr;         // [B][H][splits][d + 2]: sums, maximum, sum of weights, a float each
  uint32_t tag = 0;
  int patience = 1;                 // polls for words before this workgroup does something else
};
// LDS of the early rows: by iteration and tensor (qu, U, kc, vc, gates) 1 KB per wave
constexpr int kEarly = 2;
constexpr int kEarlyTensor = kThreads * 16, kEarlyIteration = 5 * kEarlyTensor;
extern __shared__ __attribute__((aligned(16))) unsigned char castle_early[];
__device__ __forceinline__ unsigned char* early_rows(int n, int lane) { return castle_early + n * kEarlyIteration + wave_id() * 1024 + lane * 16; }
// 16 bytes per lane from memory to consecutive places in LDS
template <bool ONCE> __device__ __forceinline__ void load_lds16(const void* from, unsigned char* to) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from, (__attribute__((address_space(3))) void*)to, 16, 0, ONCE ? 2 : 0);
}
template <typename T> constexpr int kPerWord = 4 / (int)sizeof(T);
__device__ __forceinline__ void store_word(uint64_t* p, uint32_t payload, uint32_t tag) {
  __hip_atomic_store(p, (uint64_t)tag << 32 | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// element i of a row of words from lane i (of consecutive lanes); 16-bit elements leave in pairs
template <typename T> __device__ __forceinline__ void put_word(uint64_t* row, int i, float v, uint32_t tag) {
  if constexpr (sizeof(T) == 4) {
    store_word(row + i, __builtin_bit_cast(uint32_t, v), tag);
  } else {
    const float w = __shfl_xor(v, 1);
    if (i % 2 == 0) store_word(row + i / 2, __builtin_bit_cast(uint32_t, vec<T, 2>{(T)v, (T)w}), tag);
  }
}
// N 16-byte pieces (four words each) per lane, zeros for a null pointer.  False if after `patience` polls (of about a microsecond, at least one) a word
// of the wave's lanes still does not carry the tag.
constexpr int kPatience = 64, kTries = 1 << 19;   // of a job whose operands do not come, polls each: some tens of seconds, where something else is broken
template <typename T, int N> __device__ __forceinline__ bool wait_words(const uint64_t* const (&p)[N], uint32_t tag, int patience, vec<T, elem_traits<T>::vec16> (&x)[N]) {
  for (int polls = 0; polls < patience; ++polls) {
    bool there = true;
#pragma unroll
    for (int n = 0; n < N; ++n) {
      uint64_t w[4] = {};
      if (p[n] != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = __hip_atomic_load(p[n] + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int e = 0; e < 4; ++e) there = there && (uint32_t)(w[e] >> 32) == tag;
      }
      x[n] = __builtin_bit_cast(vec<T, elem_traits<T>::vec16>, vec<uint32_t, 4>{(uint32_t)w[0], (uint32_t)w[1], (uint32_t)w[2], (uint32_t)w[3]});
    }
    if (__builtin_amdgcn_ballot_w64(!there) == 0) return true;
    __builtin_amdgcn_s_sleep(1);
  }
  return false;
}

// rows of a split: whole iterations of a workgroup
__device__ __forceinline__ int split_rows(int t, int splits, int rows_per_iteration) {
  return ((t + splits - 1) / splits + rows_per_iteration - 1) / rows_per_iteration * rows_per_iteration;
}

// A group of LPR = d / V lanes owns one cache row per iteration.  (Workgroups of 16 waves, so that a head needs no
// split and no merge, are slower throughout: 23.1 against 21.7 us for a layer step of 16 x 8 heads of 540 rows.)
//
// On three of four steps no lookahead key is written, and then none is formed either: qc . U_k of the completed key is
// qc . U_k of the stored one plus a gate times qc . vu for every pending token, which is one number per token and
// head.  (180 vector instructions per row and lane with the completed key in registers, 110 without: at 16 x 8 heads x
// 540 rows they took as long as the memory.)
//
// WORDS: a job of a launch that does the whole layer step (decode_layer_kernel below).  The token's pieces come as tagged
// words, waited for behind the requests for the first rows, and the output leaves as such; ready(whether they came) says
// whether the job goes on (if not, nothing has been written).
//
// ALIKE: the six token views have strides in common, and so have the four caches.  Formed for each view by itself, the addresses
// were 350 scalar instructions in front of the first request, most of a microsecond.
template <typename T, int HD, bool UH, bool ONCE, bool WORDS, bool ALIKE, typename G, typename F>
__device__ __forceinline__ bool stream_job(const DecodeArgs& a, int split, int bh, const TokenWords& words, G&& begin, F&& ready) {
  constexpr int V = elem_traits<T>::vec16;   // elements per 16-byte lane load
  constexpr int LPR = HD / V;                // lanes per row
  constexpr int RPI = kThreads / LPR;        // rows per workgroup iteration
  constexpr int NW = kThreads / 64;
  typedef vec<T, V> vt;
  __shared__ float s_acc[NW + (WORDS ? 1 : 0)][HD + 2];
  __shared__ float s_vu[kDecodeDefer + 1][HD];   // vu of the pending tokens by ring slot and of the new one, for steps that write U

  const int b = bh / a.H, h = bh % a.H;
  const int tid = threadIdx.x;
  const int grp = tid / LPR, sub = tid % LPR;
  // the counts of a replayed graph: on their way while the requests below are formed
  int t = a.t_dev != nullptr ? *a.t_dev : a.t;
  const int base0 = a.base0_dev != nullptr ? *a.base0_dev : a.base0;
  const int64_t tok_at = (int64_t)b * a.ku.sb + (int64_t)h * a.ku.sh, cache_at = (int64_t)b * a.U.sb + (int64_t)h * a.U.sh;
  auto tok = [&](const View4& v) __attribute__((always_inline)) {   // this lane's piece of the token
    return reinterpret_cast<const vt*>((ALIKE ? reinterpret_cast<T*>(v.ptr) + tok_at : view_row<T>(v, b, h, 0)) + sub * V);
  };
  auto cached = [&](const View4& v, int k) __attribute__((always_inline)) {   // and of a cached row
    return reinterpret_cast<vt*>((ALIKE ? reinterpret_cast<T*>(v.ptr) + cache_at + (int64_t)k * a.U.sl : view_row<T>(v, b, h, k)) + sub * V);
  };
  // All loads of the start go out together, the small ones first (they are waited for first): the token's pieces and the whole ring
  // of pending vu pieces, which do not need the row count, then the rows of the first iteration.
  vt tku, tvu, tqc;
  if constexpr (!WORDS) {
    tku = *tok(a.ku);
    tvu = *tok(a.vu);
    tqc = *tok(a.qc);
  }
  const bool deferred = a.pend_vu.ptr != nullptr;
  vt tpv[kDecodeDefer];
#pragma unroll
  for (int sl = 0; sl < kDecodeDefer; ++sl) {
#pragma unroll
    for (int e = 0; e < V; ++e) tpv[sl][e] = (T)0.f;
    if (deferred) tpv[sl] = *reinterpret_cast<const vt*>(view_row<T>(a.pend_vu, b, h, sl) + sub * V);
  }
  const bool in_range = t >= 0 && t < a.capacity;
  if (!in_range) t = 0;   // only with a device-side count: no rows, nothing is appended
  // rows of this workgroup: [r0, r1), whole iterations of RPI rows.  With WORDS the last split has none (unless it is the only
  // one): it has the appended row to see to, and the partial results of the others.
  const int with_rows = WORDS && a.splits > 1 ? a.splits - 1 : a.splits;
  const int per = split_rows(t, with_rows, RPI);
  const int r0 = split * per;
  const int r1 = min(t, r0 + per);
  // deferred write-back: how many tokens are pending, and whether this step writes U
  const int pbase = deferred ? decode_base(base0, t) : t;
  const int np = t - pbase;                                        // 0 .. kDecodeDefer - 1
  const bool write_u = !deferred || (t + 1) % kDecodeDefer == 0;
  const bool owner = split == (WORDS ? a.splits - 1 : t > 0 ? (t - 1) / per : 0);   // of the appended row
  // The row pieces of the next iteration are requested before the current one is processed.  While the token is
  // still being projected (WORDS) those of the first `early` iterations are on their way too, straight into LDS: a lane reads
  // back what it asked for.
  vt nq, nu, nk, nv;
  vec<float, 4> ng = {0.f, 0.f, 0.f, 0.f};
  constexpr int early = WORDS ? kEarly : 0;
  float* const gbase = deferred ? reinterpret_cast<float*>(a.pend_gate.ptr) + (int64_t)b * a.pend_gate.sb + (int64_t)h * a.pend_gate.sh : nullptr;
  // ONCE: past what the last-level cache (256 MB) holds of the loop this step belongs to, keeping rows in it only drives out the
  // weights and what else could stay (a layer step of 16 x 8 heads x 540 rows, one of 12 layers: 21.8 -> 19.9 us; with 6
  // layers, 212 MB, 18.7 -> 19.6)
  auto read = [](auto p) __attribute__((always_inline)) {
    if constexpr (ONCE) return __builtin_nontemporal_load(p);
    else return *p;
  };
  auto request = [&](int k) __attribute__((always_inline)) {
    if (k < r1) {
      nq = read(cached(a.qu_cache, k));
      nu = read(cached(a.U, k));
      nk = read(cached(a.kc_cache, k));
      nv = read(cached(a.vc_cache, k));
      if (np > 0) ng = read(reinterpret_cast<const vec<float, 4>*>(gbase + (int64_t)k * kDecodeDefer));
    }
  };
  if constexpr (WORDS) {
    for (int n = 0; n < early; ++n) {
      const int k = r0 + grp + n * RPI;
      if (k < r1) {
        unsigned char* const to = early_rows(n, 0);
        load_lds16<ONCE>(cached(a.qu_cache, k), to);
        load_lds16<ONCE>(cached(a.U, k), to + kEarlyTensor);
        load_lds16<ONCE>(cached(a.kc_cache, k), to + 2 * kEarlyTensor);
        load_lds16<ONCE>(cached(a.vc_cache, k), to + 3 * kEarlyTensor);
        if (np > 0) load_lds16<ONCE>(gbase + (int64_t)k * kDecodeDefer, to + 4 * kEarlyTensor);
      }
    }
  }
  request(r0 + grp + early * RPI);
  __builtin_amdgcn_sched_barrier(0);
  const float c1 = a.scale * kLog2e;
  vt tkc, tqu, tvc;
  int pend_j[kDecodeDefer];   // the token in a ring slot, or -1: a row k has a gate for token j if k < j
#pragma unroll
  for (int sl = 0; sl < kDecodeDefer; ++sl) {
    const int j = pbase + ((sl - pbase % kDecodeDefer + kDecodeDefer) % kDecodeDefer);   // the token that would sit in this slot
    pend_j[sl] = deferred && j < t ? j : -1;
  }
  if constexpr (WORDS) {
    begin();
    const uint64_t* w = words.proj + ((int64_t)b * 6 * a.H + h) * (HD / kPerWord<T>) + sub * 4;   // parts qu, ku, vu, qc, kc, vc
    const int64_t part = (int64_t)a.H * (HD / kPerWord<T>);
    vt got[6];
    const uint64_t* const need[6] = {w + part, w + 2 * part, w + 3 * part, owner ? w + 4 * part : nullptr, owner ? w : nullptr, owner ? w + 5 * part : nullptr};
    if (!ready(wait_words<T>(need, words.tag, words.patience, got))) return false;
    tku = got[0]; tvu = got[1]; tqc = got[2];
    if (owner) { tkc = got[3]; tqu = got[4]; tvc = got[5]; }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the early rows are in LDS (requested in front of the words, they came first)
  }
#pragma unroll
  for (int sl = 0; sl < kDecodeDefer; ++sl)
    if (pend_j[sl] < 0) {   // whatever an empty slot holds
#pragma unroll
      for (int e = 0; e < V; ++e) tpv[sl][e] = (T)0.f;
    }
  float ku[V], qc[V], acc[V], m = kLowest, l = 0.f;   // ku, qc times c1: products come out in log2 units
  float cvu[kDecodeDefer], cvu_t;                       // c1 qc . vu of the pending tokens and of the new one
  const int slot_t = t % kDecodeDefer;
  {
    float vu[V];
#pragma unroll
    for (int e = 0; e < V; ++e) {
      ku[e] = (float)tku[e];
      vu[e] = (float)tvu[e];
      qc[e] = (float)tqc[e];
      acc[e] = 0.f;
    }
    if (a.rotary) {   // the new token sits at position t
#pragma unroll
      for (int e = 0; e < V / 2; ++e) {
        const int pair = sub * (V / 2) + e;
        CASTLE_ROPE_PAIR(ku[2 * e], ku[2 * e + 1], (float)t, pair, HD, false);
        CASTLE_ROPE_PAIR(vu[2 * e], vu[2 * e + 1], (float)t, pair, HD, false);
        CASTLE_ROPE_PAIR(qc[2 * e], qc[2 * e + 1], (float)t, pair, HD, false);
      }
    }
    cvu_t = 0.f;
#pragma unroll
    for (int e = 0; e < V; ++e) {
      ku[e] *= c1;
      qc[e] *= c1;
      cvu_t = __builtin_fmaf(qc[e], vu[e], cvu_t);
    }
    cvu_t = group_sum<LPR>(cvu_t);
#pragma unroll
    for (int sl = 0; sl < kDecodeDefer; ++sl) {
      float c = 0.f;
#pragma unroll
      for (int e = 0; e < V; ++e) c = __builtin_fmaf(qc[e], (float)tpv[sl][e], c);
      cvu[sl] = group_sum<LPR>(c);
    }
    if (write_u && grp == 0) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
#pragma unroll
        for (int sl = 0; sl < kDecodeDefer; ++sl) s_vu[sl][sub * V + e] = (float)tpv[sl][e];
        s_vu[kDecodeDefer][sub * V + e] = vu[e];
      }
    }
  }

  auto rows = [&](auto writes) __attribute__((always_inline)) {
    int n = 0;
    for (int k = r0 + grp; k < r1; k += RPI, ++n) {
      vt cq = nq, cu = nu, ck = nk, cv = nv;
      vec<float, 4> g4 = ng;
      if (WORDS && n < early) {
        const unsigned char* const from = early_rows(n, lane_id());
        cq = *reinterpret_cast<const vt*>(from);
        cu = *reinterpret_cast<const vt*>(from + kEarlyTensor);
        ck = *reinterpret_cast<const vt*>(from + 2 * kEarlyTensor);
        cv = *reinterpret_cast<const vt*>(from + 3 * kEarlyTensor);
        g4 = *reinterpret_cast<const vec<float, 4>*>(from + 4 * kEarlyTensor);   // (not looked at without pending tokens)
      } else {
        request(k + RPI);
      }
      float dg = 0.f, dsc = 0.f, dsu = 0.f;
#pragma unroll
      for (int e = 0; e < V; ++e) {
        dg = __builtin_fmaf((float)cq[e], ku[e], dg);
        dsc = __builtin_fmaf((float)ck[e], qc[e], dsc);
      }
      const float gate = sigmoid_l2(group_sum<LPR>(dg));
      // pending sources j > k first (none unless the write-back is deferred): their gates were formed by the steps
      // that appended them and wait in the row's side array (rows appended inside the window have none for earlier tokens)
      float gj[kDecodeDefer];
#pragma unroll
      for (int sl = 0; sl < kDecodeDefer; ++sl) gj[sl] = k < pend_j[sl] ? g4[sl] : 0.f;
      if constexpr (decltype(writes)::value) {
        float uk[V];
        u_unpack<T, V, UH>(cu, uk);
        asm volatile("" ::: "memory");   // s_vu is read again for every row: held in registers it would cost 40 of them
#pragma unroll
        for (int e = 0; e < V; ++e) {
#pragma unroll
          for (int sl = 0; sl < kDecodeDefer; ++sl) uk[e] = __builtin_fmaf(gj[sl], s_vu[sl][sub * V + e], uk[e]);
          uk[e] = __builtin_fmaf(gate, s_vu[kDecodeDefer][sub * V + e], uk[e]);
        }
        // the lookahead key as later steps will see it: the stored (rounded) one
        const vt unew = u_pack<T, V, UH>(uk);
        *cached(a.U, k) = unew;
        u_unpack<T, V, UH>(unew, uk);
#pragma unroll
        for (int e = 0; e < V; ++e) dsu = __builtin_fmaf(qc[e], uk[e], dsu);
        dsu = group_sum<LPR>(dsu);
      } else {
        if constexpr (UH) {
          const vec<fp16_t, V> u = __builtin_bit_cast(vec<fp16_t, V>, cu);
#pragma unroll
          for (int e = 0; e < V; ++e) dsu = __builtin_fmaf((float)u[e], qc[e], dsu);
          dsu = group_sum<LPR>(dsu) * kUHalfUnscale;
        } else {
#pragma unroll
          for (int e = 0; e < V; ++e) dsu = __builtin_fmaf((float)cu[e], qc[e], dsu);
          dsu = group_sum<LPR>(dsu);
        }
#pragma unroll
        for (int sl = 0; sl < kDecodeDefer; ++sl) dsu = __builtin_fmaf(gj[sl], cvu[sl], dsu);
        dsu = __builtin_fmaf(gate, cvu_t, dsu);
        if (sub == 0) gbase[(int64_t)k * kDecodeDefer + slot_t] = gate;   // the new token stays pending: its gate for this row
      }
      const float x = group_sum<LPR>(dsc) - dsu * sigmoid_l2(dsu);   // score in log2 units
      const float mn = fmaxf(m, x);
      const float al = fast_exp2(m - mn), p_ = fast_exp2(x - mn);
      l = l * al + p_;
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] = __builtin_fmaf(p_, (float)cv[e], acc[e] * al);
      m = mn;
    }
  };
  if (write_u) {
    __syncthreads();   // s_vu
    rows(std::true_type());
  } else {
    rows(std::false_type());
  }
  // The owner takes row t too: U_t = 0, so its lookahead term is silu(0) = 0, and appends the new rows.  No workgroup of this
  // launch looks at row t or the ring slot of token t.
  if (owner && grp == 0) {
    if constexpr (!WORDS) {
      tkc = *tok(a.kc);
      tqu = *tok(a.qu);
      tvc = *tok(a.vc);
    }
    float kct[V], qut[V], vut[V];
#pragma unroll
    for (int e = 0; e < V; ++e) { kct[e] = (float)tkc[e]; qut[e] = (float)tqu[e]; vut[e] = (float)tvu[e]; }
    if (a.rotary) {
#pragma unroll
      for (int e = 0; e < V / 2; ++e) {
        const int pair = sub * (V / 2) + e;
        CASTLE_ROPE_PAIR(kct[2 * e], kct[2 * e + 1], (float)t, pair, HD, false);
        CASTLE_ROPE_PAIR(qut[2 * e], qut[2 * e + 1], (float)t, pair, HD, false);
        CASTLE_ROPE_PAIR(vut[2 * e], vut[2 * e + 1], (float)t, pair, HD, false);
      }
    }
    float x = 0.f;
#pragma unroll
    for (int e = 0; e < V; ++e) x = __builtin_fmaf(qc[e], kct[e], x);
    x = group_sum<LPR>(x);
    const float mn = fmaxf(m, x);
    const float al = fast_exp2(m - mn), p_ = fast_exp2(x - mn);
    l = l * al + p_;
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = __builtin_fmaf(p_, (float)tvc[e], acc[e] * al);
    m = mn;
    if (in_range) {
      vt z, q, kk, p;
#pragma unroll
      for (int e = 0; e < V; ++e) { z[e] = (T)0.f; q[e] = (T)qut[e]; kk[e] = (T)kct[e]; p[e] = (T)vut[e]; }
      *cached(a.U, t) = z;
      *cached(a.qu_cache, t) = q;
      *cached(a.kc_cache, t) = kk;
      *cached(a.vc_cache, t) = tvc;
      if (deferred) *reinterpret_cast<vt*>(view_row<T>(a.pend_vu, b, h, slot_t) + sub * V) = p;   // joins the pending sources
    }
  }
  // merge the row groups of a wave in registers, then the waves through LDS
  {
    const auto largest = [](float x, float y) { return fmaxf(x, y); };
    const auto sum = [](float x, float y) { return x + y; };
    const float M = fold_groups<LPR>(m, largest);
    const float w = fast_exp2(m - M);
    l = fold_groups<LPR>(l * w, sum);
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = fold_groups<LPR>(acc[e] * w, sum);
    m = M;
  }
  const int wave = tid / 64;
  if ((tid & 63) < LPR) {
#pragma unroll
    for (int e = 0; e < V; ++e) s_acc[wave][sub * V + e] = acc[e];
    if (sub == 0) { s_acc[wave][HD] = m; s_acc[wave][HD + 1] = l; }
  }
  __syncthreads();
  float out = 0.f, M = kLowest, lsum = 0.f;
  if (tid < HD) {
#pragma unroll
    for (int r = 0; r < NW; ++r) M = fmaxf(M, s_acc[r][HD]);
#pragma unroll
    for (int r = 0; r < NW; ++r) {
      const float w = fast_exp2(s_acc[r][HD] - M);
      out = __builtin_fmaf(w, s_acc[r][tid], out);
      lsum = __builtin_fmaf(w, s_acc[r][HD + 1], lsum);
    }
  }
  constexpr int EPL = (HD + 63) / 64;
  const int lane = tid & 63;
  if constexpr (WORDS) {
    uint64_t* const row = words.merged + (int64_t)bh * (HD / kPerWord<T>);
    if (a.splits == 1) {
      if (tid < HD) put_word<T>(row, tid, out / lsum, words.tag);
      return true;
    }
    uint64_t* const parts = words.part + (int64_t)bh * a.splits * (HD + 2);
    if (split < a.splits - 1) {
      uint64_t* const p = parts + (int64_t)split * (HD + 2);
      if (tid < HD) store_word(p + tid, __builtin_bit_cast(uint32_t, out), words.tag);
      if (tid < 2) store_word(p + HD + tid, __builtin_bit_cast(uint32_t, tid == 0 ? M : lsum), words.tag);
      return true;
    }
    // The last split's workgroup waits for the others (jobs in front of it) and merges: wave w takes every NW-th partial.  What does not come makes the
    // result NaN.
    constexpr int SU = 4;   // of them in flight
    float m_w = kLowest, l_w = 0.f, a_w[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) a_w[e] = 0.f;
    for (int s0 = wave; s0 < a.splits - 1; s0 += SU * NW) {
      float v[SU][EPL + 2];
      for (int polls = 0;; ++polls) {
        bool there = true;
#pragma unroll
        for (int u = 0; u < SU; ++u) {
          const int s = s0 + u * NW;
#pragma unroll
          for (int e = 0; e < EPL + 2; ++e) v[u][e] = e == EPL ? kLowest : 0.f;   // beyond the splits: nothing to add
          if (s < a.splits - 1) {
#pragma unroll
            for (int e = 0; e < EPL + 2; ++e) {
              const int n = e < EPL ? lane + 64 * e : HD + e - EPL;
              if (n >= HD + 2) continue;   // (lanes beyond a short row read the statistics once more)
              const uint64_t w = __hip_atomic_load(parts + (int64_t)s * (HD + 2) + n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              there = there && (uint32_t)(w >> 32) == words.tag;
              v[u][e] = __builtin_bit_cast(float, (uint32_t)w);
            }
          }
        }
        if (__builtin_amdgcn_ballot_w64(!there) == 0) break;
        if (polls == kPatience * kTries) { l_w = __builtin_nanf(""); break; }
        __builtin_amdgcn_s_sleep(1);
      }
#pragma unroll
      for (int u = 0; u < SU; ++u) {
        const float mn = fmaxf(m_w, v[u][EPL]), wo = fast_exp2(m_w - mn), wn = fast_exp2(v[u][EPL] - mn);
        l_w = l_w * wo + wn * v[u][EPL + 1];
#pragma unroll
        for (int e = 0; e < EPL; ++e) a_w[e] = a_w[e] * wo + wn * v[u][e];
        m_w = mn;
      }
    }
    __syncthreads();   // s_acc is read
#pragma unroll
    for (int e = 0; e < EPL; ++e)
      if (lane + 64 * e < HD) s_acc[wave][lane + 64 * e] = a_w[e];
    if (lane == 0) { s_acc[wave][HD] = m_w; s_acc[wave][HD + 1] = l_w; }
    if (tid < HD) s_acc[NW][tid] = out;
    if (tid == 0) { s_acc[NW][HD] = M; s_acc[NW][HD + 1] = lsum; }
    __syncthreads();
    if (tid < HD) {
      float top = kLowest, o = 0.f, l_all = 0.f;
#pragma unroll
      for (int r = 0; r <= NW; ++r) top = fmaxf(top, s_acc[r][HD]);
#pragma unroll
      for (int r = 0; r <= NW; ++r) {
        const float w = fast_exp2(s_acc[r][HD] - top);
        o = __builtin_fmaf(w, s_acc[r][tid], o);
        l_all = __builtin_fmaf(w, s_acc[r][HD + 1], l_all);
      }
      put_word<T>(row, tid, o / l_all, words.tag);
    }
    return true;
  }
  if (tid < HD) {
    if (a.splits == 1) {
      if (in_range) view_row<T>(a.out, b, h, 0)[tid] = (T)(out / lsum);
    } else {
      agent_store(part_acc(a, bh, split, HD) + tid, out);
      if (tid == 0) { agent_store(part_stat(a, bh, split, HD), M); agent_store(part_stat(a, bh, split, HD) + 1, lsum); }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
  }
  if (a.arrivals == nullptr || a.splits == 1) return true;
  __syncthreads();
  __shared__ int s_last;
  if (tid == 0) s_last = __hip_atomic_fetch_add(a.arrivals + bh, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == a.splits - 1;
  __syncthreads();
  if (!s_last || !in_range) return true;
  // the last split: lane s of every wave holds the statistics of split s (at most 64), a wave sums every fourth partial
  const float ms = lane < a.splits ? agent_load(part_stat(a, bh, lane, HD)) : -INFINITY;
  const float ls = lane < a.splits ? agent_load(part_stat(a, bh, lane, HD) + 1) : 0.f;
  float sum[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) sum[e] = 0.f;
  constexpr int SU = 4;   // partials of a wave in flight
  float wgt = 0.f;
  lsum = 0.f;
  for (int s0 = wave; s0 < a.splits; s0 += SU * NW) {
    float v[SU][EPL];
#pragma unroll
    for (int u = 0; u < SU; ++u)
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        const int s = s0 + u * NW, n = lane + 64 * e;
        v[u][e] = s < a.splits && n < HD ? agent_load(part_acc(a, bh, s, HD) + n) : 0.f;
      }
    if (s0 == wave) {   // the statistics arrive with the first partials
      M = ms;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) M = fmaxf(M, __shfl_xor(M, o));
      wgt = ms == -INFINITY ? 0.f : fast_exp2(ms - M);
      lsum = wgt * ls;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) lsum += __shfl_xor(lsum, o);
    }
#pragma unroll
    for (int u = 0; u < SU; ++u) {
      const float w = __shfl(wgt, (s0 + u * NW) & 63);   // 0 for lanes beyond the splits
#pragma unroll
      for (int e = 0; e < EPL; ++e) sum[e] = __builtin_fmaf(w, v[u][e], sum[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < EPL; ++e)
    if (lane + 64 * e < HD) s_acc[wave][lane + 64 * e] = sum[e];
  if (lane == 0 && wave == 0) s_acc[0][HD] = lsum;   // wave 0 has split 0, so it has formed the sum
  __syncthreads();
  if (tid < HD) {
    float o = 0.f;
#pragma unroll
    for (int r = 0; r < NW; ++r) o += s_acc[r][tid];
    view_row<T>(a.out, b, h, 0)[tid] = (T)(o / s_acc[0][HD]);
  }
  return true;
}
template <typename T, int HD, bool UH, bool ONCE, bool ALIKE>
__global__ __launch_bounds__(kThreads, 4) void decode_stream_kernel(DecodeArgs a) {
  stream_job<T, HD, UH, ONCE, false, ALIKE>(a, blockIdx.x, blockIdx.y, TokenWords(), [] {}, [] { return true; });
}

// One wave per (b, h): merges the split partials into the attention output.
template <typename T, int HD>
__global__ __launch_bounds__(64) void decode_finish_kernel(DecodeArgs a) {
  constexpr int EPL = (HD + 63) / 64;   // elements per lane
  const int bh = blockIdx.x, b = bh / a.H, h = bh % a.H;
  const int lane = threadIdx.x;
  const int t = a.t_dev != nullptr ? *a.t_dev : a.t;
  if (t < 0 || t >= a.capacity) return;   // only reachable with a device-side count: the cache is full
  // statistics of the partials: lane s holds split s (at most 64 splits), so the loads of all
  // splits are in flight together instead of one dependent load per loop iteration
  float ms_l = -INFINITY, ls_l = 0.f;
  if (lane < a.splits) {
    const vec<float, 2> st = *reinterpret_cast<const vec<float, 2>*>(part_stat(a, bh, lane, HD));
    ms_l = st[0];
    ls_l = st[1];
  }
  float M = ms_l;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) M = fmaxf(M, __shfl_xor(M, o));
  const float w_l = (ms_l == -INFINITY) ? 0.f : fast_exp2(ms_l - M);
  float lsum = w_l * ls_l;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) lsum += __shfl_xor(lsum, o);
  float o[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) o[e] = 0.f;
  constexpr int SU = 8;   // partial rows loaded per batch
  for (int s0 = 0; s0 < a.splits; s0 += SU) {
    float v[SU][EPL];
#pragma unroll
    for (int u = 0; u < SU; ++u)
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        const int n = lane + 64 * e;
        v[u][e] = (s0 + u < a.splits && n < HD) ? part_acc(a, bh, s0 + u, HD)[n] : 0.f;
      }
#pragma unroll
    for (int u = 0; u < SU; ++u) {
      const float w = __shfl(w_l, (s0 + u) & 63);   // 0 for lanes beyond the splits
#pragma unroll
      for (int e = 0; e < EPL; ++e) o[e] = __builtin_fmaf(w, v[u][e], o[e]);
    }
  }
  const float inv = 1.f / lsum;
  T* out = view_row<T>(a.out, b, h, 0);
#pragma unroll
  for (int e = 0; e < EPL; ++e) {
    const int n = lane + 64 * e;
    if (n < HD) out[n] = (T)(o[e] * inv);
  }
}

// Folds the pending sources into the stored lookahead keys (rows 0 .. t-1), for a reader that wants
// the cache tensor U itself: U_k += sum over pending j > k of sigmoid(s qu_k . ku_j) vu_j.
template <typename T, int HD, bool UH>
__global__ __launch_bounds__(kThreads) void decode_flush_kernel(DecodeArgs a) {
  constexpr int V = elem_traits<T>::vec16;
  constexpr int LPR = HD / V;
  constexpr int RPI = kThreads / LPR;
  typedef vec<T, V> vt;
  const int bh = blockIdx.y, b = bh / a.H, h = bh % a.H;
  const int t = a.t;
  const int grp = threadIdx.x / LPR, sub = threadIdx.x % LPR;
  const float c1 = a.scale * kLog2e;
  const int pbase = decode_base(a.base0, t);
  float pv[kDecodeDefer][V];
#pragma unroll
  for (int sl = 0; sl < kDecodeDefer; ++sl) {
#pragma unroll
    for (int e = 0; e < V; ++e) pv[sl][e] = 0.f;
    const int j = pbase + ((sl - pbase % kDecodeDefer + kDecodeDefer) % kDecodeDefer);
    if (j < t) load_f32<T, V>(view_row<T>(a.pend_vu, b, h, sl) + sub * V, pv[sl]);
  }
  (void)c1;
  for (int k = blockIdx.x * RPI + grp; k < t; k += gridDim.x * RPI) {
    float uk[V];
    T* urow = view_row<T>(a.U, b, h, k) + sub * V;
    u_unpack<T, V, UH>(*reinterpret_cast<const vt*>(urow), uk);
    const vec<float, 4> g4 = *reinterpret_cast<const vec<float, 4>*>(
        reinterpret_cast<const float*>(a.pend_gate.ptr) + (int64_t)b * a.pend_gate.sb + (int64_t)h * a.pend_gate.sh + (int64_t)k * kDecodeDefer);
#pragma unroll
    for (int sl = 0; sl < kDecodeDefer; ++sl) {
      const int j = pbase + ((sl - pbase % kDecodeDefer + kDecodeDefer) % kDecodeDefer);
      const float gj = (j < t && j > k) ? g4[sl] : 0.f;
#pragma unroll
      for (int e = 0; e < V; ++e) uk[e] = __builtin_fmaf(gj, pv[sl][e], uk[e]);
    }
    *reinterpret_cast<vt*>(urow) = u_pack<T, V, UH>(uk);
  }
}

static bool views_alike(const DecodeArgs& a) {
  auto same = [](const View4& v, const View4& w, bool rows) { return v.sb == w.sb && v.sh == w.sh && (!rows || v.sl == w.sl); };
  return same(a.kc_cache, a.U, true) && same(a.vc_cache, a.U, true) && same(a.qu_cache, a.U, true) && same(a.qc, a.ku, false) && same(a.kc, a.ku, false) &&
         same(a.vc, a.ku, false) && same(a.qu, a.ku, false) && same(a.vu, a.ku, false);
}
template <typename T, int HD, bool UH> static void launch_stream(const DecodeArgs& a, hipStream_t stream) {
  const dim3 grid(a.splits, a.B * a.H);
  auto go = [&](auto once, auto alike) {
    hipLaunchKernelGGL((decode_stream_kernel<T, HD, UH, decltype(once)::value, decltype(alike)::value>), grid, dim3(kThreads), 0, stream, a);
  };
  const std::true_type yes;
  const std::false_type no;
  if (views_alike(a)) a.read_once ? go(yes, yes) : go(no, yes);
  else a.read_once ? go(yes, no) : go(no, no);
}
template <typename T, int HD> static int launch_decode_t(const DecodeArgs& a, hipStream_t stream) {
  {
    ProfScope ps(kSlotDecodeStream, stream);
    if constexpr (__is_same(T, bf16_t)) {
      if (a.u_half) launch_stream<T, HD, true>(a, stream);
      else launch_stream<T, HD, false>(a, stream);
    } else {
      launch_stream<T, HD, false>(a, stream);
    }
  }
  if (a.splits > 1 && a.arrivals == nullptr) {
    ProfScope ps(kSlotDecodeFinish, stream);
    hipLaunchKernelGGL((decode_finish_kernel<T, HD>), dim3(a.B * a.H), dim3(64), 0, stream, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

template <typename T, int HD> static void launch_flush_t(const DecodeArgs& a, dim3 grid, hipStream_t stream) {
  if constexpr (__is_same(T, bf16_t)) {
    if (a.u_half) { hipLaunchKernelGGL((decode_flush_kernel<T, HD, true>), grid, dim3(kThreads), 0, stream, a); return; }
  }
  hipLaunchKernelGGL((decode_flush_kernel<T, HD, false>), grid, dim3(kThreads), 0, stream, a);
}
template <typename T> static int launch_flush_d(const DecodeArgs& a, hipStream_t stream) {
  const int BH = a.B * a.H;
  int gx = (640 + BH - 1) / BH;
  if (gx > 64) gx = 64;
  const dim3 grid(gx, BH);
  switch (a.d) {
    case 16: launch_flush_t<T, 16>(a, grid, stream); break;
    case 32: launch_flush_t<T, 32>(a, grid, stream); break;
    case 64: launch_flush_t<T, 64>(a, grid, stream); break;
    case 128: launch_flush_t<T, 128>(a, grid, stream); break;
    default: return -2;
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int launch_decode_flush(const DecodeArgs& a, int dtype, hipStream_t stream) {
  switch (dtype) {
    case 0: return launch_flush_d<float>(a, stream);
    case 1: return launch_flush_d<bf16_t>(a, stream);
    case 2: return launch_flush_d<fp16_t>(a, stream);
    default: return -1;
  }
}

template <typename T> static int launch_decode_d(const DecodeArgs& a, hipStream_t stream) {
  switch (a.d) {
    case 16: return launch_decode_t<T, 16>(a, stream);
    case 32: return launch_decode_t<T, 32>(a, stream);
    case 64: return launch_decode_t<T, 64>(a, stream);
    case 128: return launch_decode_t<T, 128>(a, stream);
    default: return -2;
  }
}

int launch_decode(const DecodeArgs& a, int dtype, hipStream_t stream) {
  switch (dtype) {
    case 0: return launch_decode_d<float>(a, stream);
    case 1: return launch_decode_d<bf16_t>(a, stream);
    case 2: return launch_decode_d<fp16_t>(a, stream);
    default: return -1;
  }
}

// ---------------------------------------------------------------------------
// Out-of-place rotary embedding of one (B, H, L, d) view: dst = R(pos0 + row) src.
template <typename T, int HD>
__global__ __launch_bounds__(kThreads) void rope_kernel(View4 src, View4 dst, int H, int L, int pos0) {
  constexpr int V = elem_traits<T>::vec16;
  constexpr int VPR = HD / V;
  const int bh = blockIdx.y, b = bh / H, h = bh % H;
  const int64_t piece = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t row = piece / VPR;
  const int cv = (int)(piece % VPR);
  if (row >= L) return;
  vec<float, V> f = __builtin_convertvector(*reinterpret_cast<const vec<T, V>*>(view_row<T>(src, b, h, row) + cv * V), vec<float, V>);
#pragma unroll
  for (int e = 0; e < V / 2; ++e) CASTLE_ROPE_PAIR(f[2 * e], f[2 * e + 1], (float)(pos0 + row), cv * (V / 2) + e, HD, false);
  *reinterpret_cast<vec<T, V>*>(view_row<T>(dst, b, h, row) + cv * V) = __builtin_convertvector(f, vec<T, V>);
}

// The rows of a decode cache from a projection, one launch for its three copied tensors: qu and kc (rotated by their position
// if asked for) and vc.
struct CacheRowsArgs {
  View4 src[3], dst[3];
  int H, L, rotary;
};
template <typename T, int HD>
__global__ __launch_bounds__(kThreads) void cache_rows_kernel(CacheRowsArgs a) {
  constexpr int V = elem_traits<T>::vec16;
  constexpr int VPR = HD / V;
  const int bh = blockIdx.y, b = bh / a.H, h = bh % a.H, part = blockIdx.z;
  const int64_t piece = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t row = piece / VPR;
  const int cv = (int)(piece % VPR);
  if (row >= a.L) return;
  vec<T, V> x = *reinterpret_cast<const vec<T, V>*>(view_row<T>(a.src[part], b, h, row) + cv * V);
  if (a.rotary && part != 2) {
    vec<float, V> f = __builtin_convertvector(x, vec<float, V>);
#pragma unroll
    for (int e = 0; e < V / 2; ++e) CASTLE_ROPE_PAIR(f[2 * e], f[2 * e + 1], (float)row, cv * (V / 2) + e, HD, false);
    x = __builtin_convertvector(f, vec<T, V>);
  }
  *reinterpret_cast<vec<T, V>*>(view_row<T>(a.dst[part], b, h, row) + cv * V) = x;
}
template <typename T> static int launch_cache_rows_d(const CacheRowsArgs& a, int B, int d, hipStream_t stream) {
  const int pieces_per_row = d / elem_traits<T>::vec16;
  const dim3 grid((unsigned)(((int64_t)a.L * pieces_per_row + kThreads - 1) / kThreads), B * a.H, 3);
  switch (d) {
    case 16: hipLaunchKernelGGL((cache_rows_kernel<T, 16>), grid, dim3(kThreads), 0, stream, a); break;
    case 32: hipLaunchKernelGGL((cache_rows_kernel<T, 32>), grid, dim3(kThreads), 0, stream, a); break;
    case 64: hipLaunchKernelGGL((cache_rows_kernel<T, 64>), grid, dim3(kThreads), 0, stream, a); break;
    case 128: hipLaunchKernelGGL((cache_rows_kernel<T, 128>), grid, dim3(kThreads), 0, stream, a); break;
    default: return -2;
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
int launch_cache_rows(const View4 (&src)[3], const View4 (&dst)[3], int B, int H, int L, int d, int dtype, int rotary, hipStream_t stream) {
  const CacheRowsArgs a = {{src[0], src[1], src[2]}, {dst[0], dst[1], dst[2]}, H, L, rotary};
  switch (dtype) {
    case 0: return launch_cache_rows_d<float>(a, B, d, stream);
    case 1: return launch_cache_rows_d<bf16_t>(a, B, d, stream);
    case 2: return launch_cache_rows_d<fp16_t>(a, B, d, stream);
    default: return -1;
  }
}

template <typename T> static int launch_rope_d(const View4& src, const View4& dst, int B, int H, int L, int d, int pos0, hipStream_t stream) {
  const int pieces_per_row = d / elem_traits<T>::vec16;
  const dim3 grid((unsigned)(((int64_t)L * pieces_per_row + kThreads - 1) / kThreads), B * H);
  switch (d) {
    case 16: hipLaunchKernelGGL((rope_kernel<T, 16>), grid, dim3(kThreads), 0, stream, src, dst, H, L, pos0); break;
    case 32: hipLaunchKernelGGL((rope_kernel<T, 32>), grid, dim3(kThreads), 0, stream, src, dst, H, L, pos0); break;
    case 64: hipLaunchKernelGGL((rope_kernel<T, 64>), grid, dim3(kThreads), 0, stream, src, dst, H, L, pos0); break;
    case 128: hipLaunchKernelGGL((rope_kernel<T, 128>), grid, dim3(kThreads), 0, stream, src, dst, H, L, pos0); break;
    default: return -2;
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

int launch_rope(const View4& src, const View4& dst, int B, int H, int L, int d, int dtype, int pos0, hipStream_t stream) {
  switch (dtype) {
    case 0: return launch_rope_d<float>(src, dst, B, H, L, d, pos0, stream);
    case 1: return launch_rope_d<bf16_t>(src, dst, B, H, L, d, pos0, stream);
    case 2: return launch_rope_d<fp16_t>(src, dst, B, H, L, d, pos0, stream);
    default: return -1;
  }
}

// ---------------------------------------------------------------------------
// y[M, N] = x[M, K] w[N, K]^T for the few rows of a decode step (M = batch): the two projections
// around the cached step (lookahead_keys_attention.py:99, 209 with seq_len == 1).
//
// What bounds it is latency: a launch, one trip to memory for the weights, one reduction.  So every
// 16-column slice of the output has a workgroup of its own (N = 512 then puts 32 CUs on the weights), its
// waves split K so finely that all operand loads of a wave are in flight at once (straight from global
// memory: rows of x and w are K-contiguous, which is the MFMA operand layout), and the partial tiles are
// summed through LDS.  Against 32-column slices and 8 waves throughout, replayed from a graph, 16 rows: K 2048 ->
// N 512 8.6 -> 5.6 us, 512 -> 3072 with the norm 5.4 -> 4.0, 512 -> 2048 with norm and GELU 5.1 -> 3.5, 512 -> 512
// 3.5 -> 2.7 (an empty launch takes about 2).
//
// Optional work around the product (all of it per output row, so it costs one pass less each):
//   norm_w   RMS normalisation of the x rows in front: y = ((x / rms(x)) * norm_w) w^T.  The weight
//            goes into the operand, the 1 / rms factor (a per-row scalar) onto the accumulated sum;
//            the sums of squares are collected from the fragments the product loads anyway.
//   act      1: GELU (erf form) of the sum
//   res      a tensor of the output's shape added at the end
struct LinearArgs {
  const void *x, *w;
  void* y;
  int M, N, K;
  int64_t ldx, ldw, ldy;
  const void* norm_w;
  float eps;
  int act;
  const void* res;
  int64_t ldr;
  int rows, cols;   // of the output that a workgroup takes: at most 16 MT, 16 NT
  int* clear;   // clear_n words set to zero for the launch behind this one
  int clear_n;
};
typedef vec<float, 4> acc4_t;
__device__ __forceinline__ void mma16(acc4_t& c, const vec<bf16_t, 8>& a, const vec<bf16_t, 8>& b) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ void mma16(acc4_t& c, const vec<fp16_t, 8>& a, const vec<fp16_t, 8>& b) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}
// fp32: four 4-deep products; the contraction index of slot e on lane group g is 4 g + e for both operands
__device__ __forceinline__ void mma16(acc4_t& c, const vec<float, 4>& a, const vec<float, 4>& b) {
#pragma unroll
  for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], c, 0, 0, 0);
}

// MT: 16-row tiles of a workgroup; NT: 16-column tiles; W: waves; lane l holds rows / columns l % 16, contraction piece l / 16
template <typename T, int MT, int NT, int W>
__global__ __launch_bounds__(64 * W) void small_linear_kernel(LinearArgs a) {
  constexpr int V = elem_traits<T>::vec16, DEPTH = 4 * V;   // elements of a 16-byte piece, contraction depth of one step
  constexpr int MAXS = 4;                                   // steps a wave has in flight
  typedef vec<T, V> vt;
  typedef vec<float, V> vf;
  __shared__ float red[W][16 * MT][16 * NT + 1];
  __shared__ float ssq[W][16 * MT];
  const int lane = lane_id(), wave = wave_id(), c = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * a.cols, m0 = blockIdx.y * a.rows;
  const int n_end = min(a.N, n0 + a.cols), m_end = min(a.M, m0 + a.rows);
  if (blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = threadIdx.x; i < a.clear_n; i += 64 * W) a.clear[i] = 0;
  const int steps = (a.K + DEPTH - 1) / DEPTH;
  const int per = (steps + W - 1) / W;
  const int s_end = min(steps, (wave + 1) * per);
  const T* wr = static_cast<const T*>(a.w) + (int64_t)(n0 + c) * a.ldw;
  const T* norm_w = static_cast<const T*>(a.norm_w);
  acc4_t acc[MT][NT];
  float sq[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    sq[i] = 0.f;
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = acc4_t{0.f, 0.f, 0.f, 0.f};
  }
  for (int s0 = wave * per; s0 < s_end; s0 += MAXS) {
    vt fa[MAXS][MT], fb[MAXS][NT], fg[MAXS];
#pragma unroll
    for (int u = 0; u < MAXS; ++u) {
      const int kk = DEPTH * (s0 + u) + V * g;
      const bool in = s0 + u < s_end && kk < a.K;   // K is a multiple of V
#pragma unroll
      for (int e = 0; e < V; ++e) fg[u][e] = (T)0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int e = 0; e < V; ++e) fb[u][j][e] = (T)0.f;
        if (in && n0 + 16 * j + c < n_end) fb[u][j] = *reinterpret_cast<const vt*>(wr + 16 * j * a.ldw + kk);
      }
      if (norm_w != nullptr && in) fg[u] = *reinterpret_cast<const vt*>(norm_w + kk);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int row = m0 + 16 * i + c;
#pragma unroll
        for (int e = 0; e < V; ++e) fa[u][i][e] = (T)0.f;
        if (in && row < m_end) fa[u][i] = *reinterpret_cast<const vt*>(static_cast<const T*>(a.x) + (int64_t)row * a.ldx + kk);
      }
    }
    if (norm_w != nullptr) {
#pragma unroll
      for (int u = 0; u < MAXS; ++u)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const vf xv = __builtin_convertvector(fa[u][i], vf), gv = __builtin_convertvector(fg[u], vf);
#pragma unroll
          for (int e = 0; e < V; ++e) sq[i] = __builtin_fmaf(xv[e], xv[e], sq[i]);
          fa[u][i] = __builtin_convertvector(xv * gv, vt);
        }
    }
#pragma unroll
    for (int u = 0; u < MAXS; ++u)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) mma16(acc[i][j], fa[u][i], fb[u][j]);
  }
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave][16 * i + 4 * g + r][16 * j + c] = acc[i][j][r];
  if (norm_w != nullptr) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {   // the four contraction pieces of a row
      sq[i] += __shfl_xor(sq[i], 16);
      sq[i] += __shfl_xor(sq[i], 32);
      if (g == 0) ssq[wave][16 * i + c] = sq[i];
    }
  }
  __syncthreads();
#pragma unroll
  for (int o = threadIdx.x; o < 256 * MT * NT; o += 64 * W) {
    const int row = o / (16 * NT), col = o % (16 * NT);
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < W; ++v) s += red[v][row][col];
    if (norm_w != nullptr) {
      float t = 0.f;
#pragma unroll
      for (int v = 0; v < W; ++v) t += ssq[v][row];
      s *= __builtin_amdgcn_rsqf(t / (float)a.K + a.eps);
    }
    if (a.act == 1) s = 0.5f * s * (1.f + erff(s * 0.70710678f));
    if (m0 + row < m_end && n0 + col < n_end) {
      if (a.res != nullptr) s += (float)static_cast<const T*>(a.res)[(int64_t)(m0 + row) * a.ldr + n0 + col];
      static_cast<T*>(a.y)[(int64_t)(m0 + row) * a.ldy + n0 + col] = (T)s;
    }
  }
}

template <typename T> static void launch_linear_t(LinearArgs a, hipStream_t stream) {
  // 16 waves when K is long enough to give each of them two steps
  const bool wide = a.K >= 16 * 4 * elem_traits<T>::vec16 * 2;
  // Rows x columns of a workgroup: a CU draws about 40 bytes per ns, so what counts is the rows of x plus the columns of w
  // that the busiest CU reads.  Parts of a 16 x 16 matrix tile stay empty for it: K 2048 -> N 512 with 16 rows takes
  // 32 CUs of 128 KB as 16 x 16, 128 CUs of 64 KB as 8 x 8.
  int64_t best = INT64_MAX;
  for (int r = 8; r <= 32; r *= 2)
    for (int c = 8; c <= 32; c *= 2) {
      const int64_t groups = (int64_t)((a.M + r - 1) / r) * ((a.N + c - 1) / c), cost = (groups + 255) / 256 * (std::min(r, a.M) + c) * 1024 + groups / 64;
      if (cost < best) { best = cost; a.rows = r; a.cols = c; }
    }
  const int mt = a.rows > 16 ? 2 : 1, nt = a.cols > 16 ? 2 : 1;
  const dim3 grid((a.N + a.cols - 1) / a.cols, (a.M + a.rows - 1) / a.rows), block(wide ? 1024 : 512);
#define CASTLE_LINEAR(MT_, NT_, W_) hipLaunchKernelGGL((small_linear_kernel<T, MT_, NT_, W_>), grid, block, 0, stream, a)
  if (wide) {
    if (mt == 1) { if (nt == 1) CASTLE_LINEAR(1, 1, 16); else CASTLE_LINEAR(1, 2, 16); }
    else { if (nt == 1) CASTLE_LINEAR(2, 1, 16); else CASTLE_LINEAR(2, 2, 16); }
  } else {
    if (mt == 1) { if (nt == 1) CASTLE_LINEAR(1, 1, 8); else CASTLE_LINEAR(1, 2, 8); }
    else { if (nt == 1) CASTLE_LINEAR(2, 1, 8); else CASTLE_LINEAR(2, 2, 8); }
  }
#undef CASTLE_LINEAR
}
int launch_small_linear(const void* x, const void* w, void* y, int M, int N, int K, int64_t ldx, int64_t ldw, int64_t ldy,
                        int dtype, const void* norm_w, float eps, int act, const void* res, int64_t ldr, hipStream_t stream, int* clear, int clear_n) {
  const LinearArgs a = {x, w, y, M, N, K, ldx, ldw, ldy, norm_w, eps, act, res, ldr, 0, 0, clear, clear_n};
  switch (dtype) {
    case 0: launch_linear_t<float>(a, stream); break;
    case 1: launch_linear_t<bf16_t>(a, stream); break;
    case 2: launch_linear_t<fp16_t>(a, stream); break;
    default: return -1;
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ---------------------------------------------------------------------------
// The whole layer step in one launch: jobs for the tiles of the projection, for the splits of the streaming pass and for the
// tiles of the output projection, one workgroup each, in that order.
//
// What bounds it is trips to memory, one after the other: arguments, weights, reduction (3.1 us until the projection is
// stored), the words of the token (2), rows and their sums (3), the partial results (2), the words of the output and the last product
// (2.5).  The streaming jobs have requested their rows and the output jobs hold their weights by the time the projection is
// done; a word takes 0.6 us from its store to a load that sees it, and a poll about one.
//
// Waiting inside a launch ends only if what is waited for runs.  Nothing is assumed about the order in which workgroups
// start: every job is claimed before it writes anything (one word per job), jobs wait for jobs in front of them only, for a
// bounded time, and a workgroup that has waited in vain claims and runs what nobody has claimed in front of its own job, first to
// last, before it tries its own again.  The first of the unfinished jobs finds all it needs, so there is always one that
// ends.  (The last split waits for the others without taking over anything, but only once all of them are claimed.)  A workgroup whose job was
// taken leaves.  The last workgroup to leave moves the tag on, so that no launch can take words or claims of another for
// its own.
// Every wait is bounded all the same (kTries).  A job that is given up at the end leaves NaN: in its words, in its part of y, and in a value row of
// its head, so that neither this step nor a later one on the cache passes for a good one.
constexpr int kExitGroups = 32, kLine = 32;   // words of a 128-byte line
constexpr int kLayerJobs = 2048;
constexpr int kLayerGroups = 3;   // workgroups of a CU
// Which steps: what one launch saves is the host's work for two more, 15 to 16 us a step with three whatever shorter kernels take; what it costs
// are the hand-overs and the smaller workgroups of the products (us a step, three / one; heads of 64 elements with 300 rows and a layer of width 512,
// 16 bit, if nothing else is said).  Ahead or level: 1 x 8 heads 16.3 / 13.0, 1 x 16 15.8 / 15.3, 4 x 8 15.6 / 13.9, 8 x 8 15.5 / 15.0, 16 x 4 15.6 / 14.6,
// 64 x 2 heads of 32 with 100 rows 15.5 / 14.1, 1 x 2 with 2500 rows 15.4 / 14.6; width 256 1 x 4 15.4 / 12.8, 16 x 4 with 100 rows 16.0 / 13.2, fp32 1 x 4 15.3 / 14.0,
// 1 x 4 with 900 rows 15.0 / 14.8, 1 x 5 15.1 / 14.9.  Not where
// - the contraction of the projection is longer than what the four waves of a job request at once, since every further round is a trip to
//   memory: width 768 4 x 12 15.7 / 16.5, 1024 8 x 16 16.3 / 20.3, 2048 16 x 4 15.6 / 20.9, 4096 1 x 4 15.8 / 21.3, fp32 512 1 x 8 15.6 / 17.2;
// - many jobs come before the output projection (layer_front): 8 x 16 with 40 rows 15.7 / 18.0, 16 x 8 with 100 15.8 / 16.2, 64 x 4 with 40
//   15.6 / 16.3, 1 x 32 16.0 / 16.5, fp32 width 256 1 x 5 with 600 rows 15.0 / 15.4, with 900 14.8 / 15.9, 1 x 16 16.7 / 20.5;
// - the merge of a head takes more than two rounds: 1 x 1 of 128 with 2900 rows 15.2 / 20.3, fp32 1 x 2 with 2500 15.1 / 17.5;
// - the cached rows take longer to read than the launches: 8 x 8 heads of 1000 rows 19.3 / 20.9;
// - the row count is on the device: replayed from a graph, a hand-over inside a launch costs what a launch does (29.1 / 29.2 with feed-forward at 1 x 8
//   heads of 300 rows, 36.5 / 37.6 at 16 x 8).
constexpr int kLayerRound = 1024;                               // bytes of the contraction
constexpr int kLayerFront16 = 512, kLayerFront32 = 176;         // jobs before the output projection: two a CU in 16 bit, two thirds of one in fp32
constexpr int kLayerSplits = 33;                                // 32 partial results, and the last split's own
constexpr int64_t kLayerCacheBytes = 10 << 20;                  // of cached rows
constexpr int layer_front(int es) { return es == 2 ? kLayerFront16 : kLayerFront32; }
struct LayerArgs {
  DecodeArgs d;
  LinearArgs in, out;
  uint32_t* control;   // tag of the last launch; workgroups gone, in all and by group, a line each; claims
  uint64_t *proj, *merged, *part;
  int n_in, n_stream, n_out, in_cols, out_cols;   // jobs; column tiles of the two products
  int patience, tries;
  bool reversed;   // the first workgroup has the last job
};
constexpr int kGone = kLine, kGoneGroup = 2 * kLine, kClaims = kGoneGroup + kExitGroups * kLine;

__device__ __forceinline__ uint32_t agent_word(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
// true if the job was free
__device__ __forceinline__ bool claim_job(uint32_t* claims, int job, uint32_t tag) {
  return __hip_atomic_exchange(claims + job, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != tag;
}
// by each wave: n jobs (at most 64) are claimed
__device__ __forceinline__ bool jobs_claimed(const uint32_t* claims, int n, uint32_t tag) {
  const bool open = lane_id() < n && agent_word(claims + min(lane_id(), n - 1)) != tag;
  return __builtin_amdgcn_ballot_w64(open) == 0;
}
// by one wave: claims the first free one of the first n jobs, -1 if there is none
__device__ __forceinline__ int take_job(uint32_t* claims, int n, uint32_t tag) {
  for (int base = 0; base < n; base += 64) {
    const int i = base + lane_id();
    unsigned long long open = __builtin_amdgcn_ballot_w64(i < n && agent_word(claims + min(i, n - 1)) != tag);
    while (open != 0) {
      const int job = base + __builtin_ctzll(open);
      int got = 0;
      if (lane_id() == 0) got = claim_job(claims, job, tag);
      if (__builtin_amdgcn_readfirstlane(got)) return job;
      open &= open - 1;
    }
  }
  return -1;
}

struct LinearLds {
  float red[kThreads / 64][16][17];
  float ssq[kThreads / 64][16];
};
__device__ __forceinline__ LinearLds& linear_lds() {
  __shared__ LinearLds lds;
  return lds;
}
// One 16 x 16 tile (or part of one) of y = x w^T, the K split over the waves as in small_linear_kernel.  WORDS_IN: x comes as words, else
// y leaves as words.  ready(whether the words came): a barrier that says whether the result may be written.
template <typename T, bool WORDS_IN, typename G, typename F>
__device__ __forceinline__ bool linear_job(const LinearArgs& a, int tile, int col_tiles, const uint64_t* xw, uint64_t* yw, uint32_t tag, int patience, G&& begin, F&& ready) {
  constexpr int V = elem_traits<T>::vec16, DEPTH = 4 * V, MAXS = 4, W = kThreads / 64;
  typedef vec<T, V> vt;
  typedef vec<float, V> vf;
  auto& red = linear_lds().red;
  auto& ssq = linear_lds().ssq;
  const int lane = lane_id(), wave = wave_id(), c = lane & 15, g = lane >> 4;
  const int n0 = tile % col_tiles * a.cols, m0 = tile / col_tiles * a.rows;
  const int n_end = min(a.N, n0 + a.cols), m_end = min(a.M, m0 + a.rows), row = m0 + c;
  const int steps = (a.K + DEPTH - 1) / DEPTH;
  const int per = (steps + W - 1) / W;
  const int s_end = min(steps, (wave + 1) * per);
  const T* wr = static_cast<const T*>(a.w) + (int64_t)(n0 + c) * a.ldw;
  const T* norm_w = static_cast<const T*>(a.norm_w);
  acc4_t acc = {0.f, 0.f, 0.f, 0.f};
  float sq = 0.f;
  vt fb[MAXS];
  auto weights = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < MAXS; ++u) {
      const int kk = DEPTH * (s0 + u) + V * g;
#pragma unroll
      for (int e = 0; e < V; ++e) fb[u][e] = (T)0.f;
      if (s0 + u < s_end && kk < a.K && n0 + c < n_end) fb[u] = *reinterpret_cast<const vt*>(wr + kk);   // K is a multiple of V
    }
  };
  weights(wave * per);
  if constexpr (WORDS_IN) begin();
  bool came = true;
  for (int s0 = wave * per; s0 < s_end; s0 += MAXS) {
    vt fa[MAXS], fg[MAXS];
    if constexpr (WORDS_IN) {
      // the first piece until it is there, then the others together: polling all of them would take 32 KB a round
      auto at = [&](int u) __attribute__((always_inline)) {
        const int kk = DEPTH * (s0 + u) + V * g;
        return s0 + u < s_end && kk < a.K && row < m_end ? xw + ((int64_t)row * a.K + kk) / kPerWord<T> : nullptr;
      };
      const uint64_t* const first[1] = {at(0)};
      const uint64_t* const rest[MAXS - 1] = {at(1), at(2), at(3)};
      vt x0[1], xr[MAXS - 1];
      came = came && wait_words<T>(first, tag, patience, x0) && wait_words<T>(rest, tag, patience, xr);
      fa[0] = x0[0];
#pragma unroll
      for (int u = 1; u < MAXS; ++u) fa[u] = xr[u - 1];
    } else {
#pragma unroll
      for (int u = 0; u < MAXS; ++u) {
        const int kk = DEPTH * (s0 + u) + V * g;
        const bool in = s0 + u < s_end && kk < a.K;
#pragma unroll
        for (int e = 0; e < V; ++e) { fa[u][e] = (T)0.f; fg[u][e] = (T)0.f; }
        if (in && norm_w != nullptr) fg[u] = *reinterpret_cast<const vt*>(norm_w + kk);
        if (in && row < m_end) fa[u] = *reinterpret_cast<const vt*>(static_cast<const T*>(a.x) + (int64_t)row * a.ldx + kk);
      }
      begin();
      if (norm_w != nullptr) {
#pragma unroll
        for (int u = 0; u < MAXS; ++u) {
          const vf xv = __builtin_convertvector(fa[u], vf), gv = __builtin_convertvector(fg[u], vf);
#pragma unroll
          for (int e = 0; e < V; ++e) sq = __builtin_fmaf(xv[e], xv[e], sq);
          fa[u] = __builtin_convertvector(xv * gv, vt);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < MAXS; ++u) mma16(acc, fa[u], fb[u]);
    weights(s0 + MAXS);
  }
  asm volatile("s_nop 15" ::: "memory");   // the loop may end right behind a product
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wave][4 * g + r][c] = acc[r];
  if (!WORDS_IN && norm_w != nullptr) {   // the four contraction pieces of a row
    sq += __shfl_xor(sq, 16);
    sq += __shfl_xor(sq, 32);
    if (g == 0) ssq[wave][c] = sq;
  }
  if (!ready(came)) return false;
  constexpr int E = WORDS_IN ? 1 : kPerWord<T>;   // columns of a thread
  const int o = threadIdx.x;
  if (o < 256 / E) {
    const int rr = o / (16 / E), col = o % (16 / E) * E;
    float s[E];
    float scale = 1.f;
    if (!WORDS_IN && norm_w != nullptr) {
      float t = 0.f;
#pragma unroll
      for (int v = 0; v < W; ++v) t += ssq[v][rr];
      scale = __builtin_amdgcn_rsqf(t / (float)a.K + a.eps);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      s[e] = 0.f;
#pragma unroll
      for (int v = 0; v < W; ++v) s[e] += red[v][rr][col + e];
      if (!WORDS_IN && norm_w != nullptr) s[e] *= scale;
    }
    if (m0 + rr < m_end && n0 + col < n_end) {
      if constexpr (WORDS_IN) {
        if (a.res != nullptr) s[0] += (float)static_cast<const T*>(a.res)[(int64_t)(m0 + rr) * a.ldr + n0 + col];
        static_cast<T*>(a.y)[(int64_t)(m0 + rr) * a.ldy + n0 + col] = (T)s[0];
      } else {
        uint32_t payload;
        if constexpr (E == 2) payload = __builtin_bit_cast(uint32_t, vec<T, 2>{(T)s[0], (T)s[1]});
        else payload = __builtin_bit_cast(uint32_t, s[0]);
        store_word(yw + ((int64_t)(m0 + rr) * a.N + n0 + col) / kPerWord<T>, payload, tag);
      }
    }
  }
  return true;
}

// what a job that is given up leaves (those of the projection wait for nothing)
template <typename T, int HD> __device__ __forceinline__ void give_up(const LayerArgs& f, int job, uint32_t tag) {
  const T nan = (T)__builtin_nanf("");
  const int tid = threadIdx.x, stream = job - f.n_in, out = stream - f.n_stream;
  if (out >= 0) {
    const int m = out / f.out_cols * f.out.rows + tid / 16, n = out % f.out_cols * f.out.cols + tid % 16;
    if (tid / 16 < f.out.rows && tid % 16 < f.out.cols && m < f.out.M && n < f.out.N) static_cast<T*>(f.out.y)[(int64_t)m * f.out.ldy + n] = nan;
    return;
  }
  const int bh = stream / f.d.splits, split = stream % f.d.splits;
  const bool last = split == f.d.splits - 1;
  if (last) {
    uint32_t payload;
    if constexpr (sizeof(T) == 4) payload = __builtin_bit_cast(uint32_t, nan);
    else payload = __builtin_bit_cast(uint32_t, vec<T, 2>{nan, nan});
    for (int i = tid; i < HD / kPerWord<T>; i += kThreads) store_word(f.merged + (int64_t)bh * (HD / kPerWord<T>) + i, payload, tag);
  } else {
    for (int i = tid; i < HD + 2; i += kThreads) store_word(f.part + (int64_t)stream * (HD + 2) + i, __builtin_bit_cast(uint32_t, __builtin_nanf("")), tag);
  }
  // of its own rows the first, of the last split the appended one
  const int row = last ? f.d.t : split * split_rows(f.d.t, f.d.splits - 1, kThreads * elem_traits<T>::vec16 / HD);
  if (last || row < f.d.t)
    for (int e = tid; e < HD; e += kThreads) view_row<T>(f.d.vc_cache, bh / f.d.H, bh % f.d.H, row)[e] = nan;
}

template <typename T, int HD, bool UH>
__global__ __launch_bounds__(kThreads, kLayerGroups) void decode_layer_kernel(LayerArgs args) {
  __shared__ int s_mine, s_came[kThreads / 64], s_job;
  const int own = args.reversed ? gridDim.x - 1 - blockIdx.x : blockIdx.x;
  uint32_t* const claims = args.control + kClaims;
  const uint32_t tag = args.control[0] + 1;
  bool claimed = false, mine = true;   // mine, of thread 0: the claim's answer
  // behind the first loads of a job: the tag is there by then, and the answer when the loads are
  auto begin = [&] __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    if (!claimed && threadIdx.x == 0) mine = claim_job(claims, own, tag);
    claimed = true;
    __builtin_amdgcn_sched_barrier(0);
  };
  enum { kTaken, kGo, kLater };   // another workgroup has the job; it may go on; something it needs is missing
  int answer = kGo;
  auto agree = [&](bool came) __attribute__((always_inline)) {
    if (threadIdx.x == 0) s_mine = mine;
    if (lane_id() == 0) s_came[wave_id()] = came;
    __syncthreads();
    bool all = true;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) all = all && s_came[w];
    answer = __builtin_amdgcn_readfirstlane(!s_mine ? kTaken : all ? kGo : kLater);
    return answer == kGo;
  };
  auto run = [&](const LayerArgs& f, int job) __attribute__((always_inline)) {
    const int stream = job - f.n_in, out = stream - f.n_stream;
    if (stream < 0) {
      linear_job<T, false>(f.in, job, f.in_cols, nullptr, f.proj, tag, f.patience, begin, agree);
    } else if (out < 0) {
      const int split = stream % f.d.splits;
      const TokenWords words = {f.proj, f.merged, f.part, tag, f.patience};
      stream_job<T, HD, UH, false, true, true>(f.d, split, stream / f.d.splits, words, begin, [&](bool came) {
        // the last split waits for the others' partial results when its own rows are done: they have to be claimed by now
        if (split == f.d.splits - 1) came = came && jobs_claimed(claims + job - split, split, tag);
        return agree(came);
      });
    } else {
      linear_job<T, true>(f.out, out, f.out_cols, f.merged, nullptr, tag, f.patience, begin, agree);
    }
  };
  run(args, own);
  int job = own;
  // The arguments are read where a job needs them: read ahead of the loop, 160 scalar and 80 vector registers spill.
  auto again = [] __attribute__((always_inline)) {
    const __attribute__((address_space(4))) LayerArgs* kernarg = (const __attribute__((address_space(4))) LayerArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(kernarg));
    return (const LayerArgs*)kernarg;
  };
  for (int tries = 0; job != own || answer == kLater; ++tries) {
    if (tries >= again()->tries) {
      if (answer == kLater) give_up<T, HD>(*again(), job, tag);
      if (job != own) give_up<T, HD>(*again(), own, tag);   // (its own waited for the one it took)
      break;
    }
    __syncthreads();   // what the last job kept in LDS is read
    if (job == own || answer != kLater) {   // (a job once taken is run until it is done)
      if (wave_id() == 0) {
        const int j = take_job(claims, own, tag);
        if (threadIdx.x == 0) s_job = j;
      }
      __syncthreads();
      job = __builtin_amdgcn_readfirstlane(s_job);
      if (job < 0) job = own;
    }
    run(*again(), job);
  }
  if (threadIdx.x == 0) {
    const int groups = min(kExitGroups, (int)gridDim.x), g = blockIdx.x % kExitGroups;
    const int members = ((int)gridDim.x - g + kExitGroups - 1) / kExitGroups;
    uint32_t* const gone = args.control + kGoneGroup + g * kLine;
    auto add = [](uint32_t* p) { return (int)__hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    auto set = [](uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    if (add(gone) == members - 1) {
      set(gone, 0);
      if (add(args.control + kGone) == groups - 1) {
        set(args.control + kGone, 0);
        set(args.control, tag);
      }
    }
  }
}

static int64_t word_count(int64_t elements, int es) { return elements * es / 4; }
int64_t decode_layer_control_bytes(int B, int H, int d, int es) {
  return (kClaims + kLayerJobs) * 4 + 8 * (word_count((int64_t)B * 6 * H * d, es) + word_count((int64_t)B * H * d, es) + (int64_t)layer_front(es) * (d + 2));
}

// Rows x columns (at most 16 x 16) of a job: small ones while that leaves no CU a second
static void pick_job_tile(LinearArgs& a) {
  a.rows = a.cols = 16;
  for (int r = 8; r <= 16; r *= 2)
    for (int c = 8; c <= 16; c *= 2) {
      const int64_t groups = (int64_t)((a.M + r - 1) / r) * ((a.N + c - 1) / c);
      if (groups <= 128 && std::min(r, a.M) + c < std::min(a.rows, a.M) + a.cols) { a.rows = r; a.cols = c; }
    }
}
template <typename T, int HD> static int launch_layer_t(const LayerArgs& f, hipStream_t stream) {
  ProfScope ps(kSlotDecodeStream, stream);
  const dim3 grid(f.n_in + f.n_stream + f.n_out), block(kThreads);
  constexpr int lds = kEarly * kEarlyIteration;
  if constexpr (__is_same(T, bf16_t)) {
    if (f.d.u_half) hipLaunchKernelGGL((decode_layer_kernel<T, HD, true>), grid, block, lds, stream, f);
    else hipLaunchKernelGGL((decode_layer_kernel<T, HD, false>), grid, block, lds, stream, f);
  } else {
    hipLaunchKernelGGL((decode_layer_kernel<T, HD, false>), grid, block, lds, stream, f);
  }
  return hipGetLastError() == hipSuccess ? 0 : -3;
}
template <typename T> static int launch_layer_d(const LayerArgs& f, hipStream_t stream) {
  switch (f.d.d) {
    case 16: return launch_layer_t<T, 16>(f, stream);
    case 32: return launch_layer_t<T, 32>(f, stream);
    case 64: return launch_layer_t<T, 64>(f, stream);
    case 128: return launch_layer_t<T, 128>(f, stream);
    default: return -2;
  }
}

// Tiles, splits and jobs of a step whose sizes are in d, in and out; false if it does not go in one launch (see kLayerRound).
static bool layer_jobs(LayerArgs& f, int es) {
  pick_job_tile(f.in);
  pick_job_tile(f.out);
  f.in_cols = (f.in.N + f.in.cols - 1) / f.in.cols;
  f.out_cols = (f.out.N + f.out.cols - 1) / f.out.cols;
  const int64_t n_in = (int64_t)f.in_cols * ((f.in.M + f.in.rows - 1) / f.in.rows), n_out = (int64_t)f.out_cols * ((f.out.M + f.out.rows - 1) / f.out.rows);
  const int64_t BH = (int64_t)f.d.B * f.d.H;
  const int rows = kThreads * 16 / (f.d.d * es) * (kEarly + 1);   // of a split: what it requests ahead of the token
  f.d.splits = (int64_t)f.d.t * (kEarly + 1) <= rows ? 1 : (f.d.t + rows - 1) / rows + 1;
  if ((int64_t)f.in.K * es > kLayerRound || 4 * BH * f.d.t * f.d.d * es > kLayerCacheBytes || f.d.splits > kLayerSplits || n_in + BH * f.d.splits > layer_front(es) ||
      n_in + BH * f.d.splits + n_out > kLayerJobs)
    return false;
  f.n_in = (int)n_in;
  f.n_out = (int)n_out;
  f.n_stream = (int)BH * f.d.splits;
  return true;
}
bool decode_layer_once_ok(int B, int H, int d, int es, int t, int dim) {
  LayerArgs f = {};
  f.d.B = B; f.d.H = H; f.d.d = d; f.d.t = t;
  f.in.M = f.out.M = B;
  f.in.N = 6 * H * d; f.in.K = dim;
  f.out.N = dim; f.out.K = H * d;
  return layer_jobs(f, es);
}

// 1: the step does not go in one launch: by its sizes, with its row count on the device, or with views whose strides differ.
int launch_decode_layer(const DecodeArgs& d, const DecodeLinear& in, const DecodeLinear& out, void* control, bool take_over, bool give_up, int dtype, hipStream_t stream) {
  const int es = dtype == 0 ? 4 : 2;
  LayerArgs f = {};
  f.d = d;
  f.in = {in.x, in.w, nullptr, in.M, in.N, in.K, in.ldx, in.ldw, 0, in.norm_w, in.eps, 0, nullptr, 0, 0, 0, nullptr, 0};
  f.out = {nullptr, out.w, out.y, out.M, out.N, out.K, 0, out.ldw, out.ldy, nullptr, 0.f, 0, out.res, out.ldr, 0, 0, nullptr, 0};
  if (d.t_dev != nullptr || !views_alike(d) || !layer_jobs(f, es)) return 1;
  f.patience = take_over || give_up ? 1 : kPatience;
  f.tries = give_up ? 0 : kTries;
  f.reversed = take_over || give_up;
  char* p = static_cast<char*>(control);
  f.control = reinterpret_cast<uint32_t*>(p);
  p += (kClaims + kLayerJobs) * 4;
  f.proj = reinterpret_cast<uint64_t*>(p);
  f.merged = f.proj + word_count((int64_t)d.B * in.N, es);
  f.part = f.merged + word_count((int64_t)d.B * out.K, es);
  switch (dtype) {
    case 0: return launch_layer_d<float>(f, stream);
    case 1: return launch_layer_d<bf16_t>(f, stream);
    case 2: return launch_layer_d<fp16_t>(f, stream);
    default: return -1;
  }
}

// ---------------------------------------------------------------------------
// One token per row from its logits (train_triton.py:56-71): keep the k largest, divide by the temperature, add
// Gumbel noise formed from the uniform numbers `u`, take the arg-max.  As separate operators (a radix top-k, its sort, a
// scatter, twice clamp / log / negate, add, arg-max) this is 15 launches and ~100 us per token around a model step of
// ~400; here one workgroup per row finds the k-th largest value by a radix select over the row (4 rounds of 256 bins,
// the row stays in L2) and takes the arg-max of what is at or above it in the same launch.
constexpr int kSampleThreads = 512;
struct SampleArgs {
  const void* logits;
  int64_t ld;
  const float* u;   // [rows][V] uniform numbers; nullptr: no noise (arg-max)
  int V, k;
  float inv_temperature;
  int64_t *out, out_ld;   // one token per row
  int64_t* out2;          // optional second copy, contiguous
};
// order-preserving map of a float to an unsigned integer; NaN above everything
__device__ __forceinline__ uint32_t float_order(float x) {
  const uint32_t b = __builtin_bit_cast(uint32_t, x);
  return x == x ? b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u) : 0xffffffffu;
}
// the same from the bits of the type itself, 16 for 16-bit types; never 0
template <typename T> __device__ __forceinline__ uint32_t type_order(T x) {
  if constexpr (sizeof(T) == 4) {
    return float_order(x);
  } else {
    const uint32_t b = __builtin_bit_cast(uint16_t, x);
    return (float)x == (float)x ? b ^ ((b >> 15) ? 0xffffu : 0x8000u) : 0xffffu;
  }
}
// the logit of a kept token with its noise
__device__ __forceinline__ float with_noise(float v, float u, float inv_temperature) {
  const float e = -logf(fmaxf(u, 1e-20f));
  return v * inv_temperature - logf(fmaxf(e, 1e-20f));
}
// the largest, the lowest index among equals; a NaN counts as the largest
__device__ __forceinline__ bool better_token(float v, int i, float w, int j) {
  return i != 0x7fffffff && (j == 0x7fffffff || (v != v ? !(w != w) || i < j : w == w && (v > w || (v == w && i < j))));
}
// A vocabulary of up to 64 E: one wave per row with E logits in each lane, no LDS and no barrier.  The k-th largest bit by bit from the
// top, each a count over the wave, 16 for 16-bit logits (16 rows of 256 bf16 logits: 7.9 us by radix rounds over 512 threads, 5.0 here).
template <typename T, int E> __global__ __launch_bounds__(64) void sample_few_kernel(SampleArgs a) {
  const int row = blockIdx.x, lane = threadIdx.x;
  const T* x = static_cast<const T*>(a.logits) + (int64_t)row * a.ld;
  T v[E];
  float u[E];
  uint32_t order[E];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = x[min(64 * e + lane, a.V - 1)];
  if (a.u != nullptr) {
#pragma unroll
    for (int e = 0; e < E; ++e) u[e] = a.u[(int64_t)row * a.V + min(64 * e + lane, a.V - 1)];
  }
#pragma unroll
  for (int e = 0; e < E; ++e) order[e] = 64 * e + lane < a.V ? type_order(v[e]) : 0;
  uint32_t kth = 0;
  for (uint32_t bit = 1u << (8 * sizeof(T) - 1); bit != 0; bit >>= 1) {
    int n = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(order[e] >= (kth | bit)));
    if (n >= a.k) kth |= bit;
  }
  int left = a.k;   // of those equal to the k-th, in index order
#pragma unroll
  for (int e = 0; e < E; ++e) left -= __builtin_popcountll(__builtin_amdgcn_ballot_w64(order[e] > kth));
  float best = -INFINITY;
  int arg = 0x7fffffff;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int i = 64 * e + lane;
    const bool equal = i < a.V && order[e] == kth;
    const unsigned long long ballot = __builtin_amdgcn_ballot_w64(equal);
    const bool kept = i < a.V && (order[e] > kth || (equal && __builtin_popcountll(ballot & ((1ull << lane) - 1)) < left));
    left -= __builtin_popcountll(ballot);
    const float z = a.u != nullptr ? with_noise((float)v[e], u[e], a.inv_temperature) : (float)v[e];
    if (kept && better_token(z, i, best, arg)) { best = z; arg = i; }
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float ob = __shfl_xor(best, o);
    const int oa = __shfl_xor(arg, o);
    if (better_token(ob, oa, best, arg)) { best = ob; arg = oa; }
  }
  if (lane == 0) {
    a.out[(int64_t)row * a.out_ld] = arg;
    if (a.out2 != nullptr) a.out2[row] = arg;
  }
}
template <typename T>
__global__ __launch_bounds__(kSampleThreads) void sample_kernel(SampleArgs a) {
  constexpr int NW = kSampleThreads / 64;
  __shared__ int hist[256];
  __shared__ int s_bin, s_left, s_taken;
  __shared__ int s_wave[NW];
  __shared__ float s_best[NW];
  __shared__ int s_arg[NW];
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const T* x = static_cast<const T*>(a.logits) + (int64_t)row * a.ld;
  // the k-th largest value: digit by digit from the top, `left` of the values with the digits found so far wanted
  uint32_t prefix = 0, mask = 0;
  int left = a.k;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int i = tid; i < 256; i += kSampleThreads) hist[i] = 0;
    __syncthreads();
    for (int i = tid; i < a.V; i += kSampleThreads) {
      const uint32_t o = float_order((float)x[i]);
      if ((o & mask) == prefix) atomicAdd(&hist[(o >> shift) & 255], 1);
    }
    __syncthreads();
    if (wave == 0) {   // suffix sums of the 256 bins, four per lane, from the highest bin down
      int h[4], sum = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) { h[e] = hist[255 - (4 * lane + e)]; sum += h[e]; }
      int above = sum;   // inclusive scan over lanes
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(above, o);
        if (lane >= o) above += y;
      }
      above -= sum;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (above < left && above + h[e] >= left) { s_bin = 255 - (4 * lane + e); s_left = left - above; }
        above += h[e];
      }
    }
    __syncthreads();
    prefix |= (uint32_t)s_bin << shift;
    mask |= 255u << shift;
    left = s_left;
    __syncthreads();
  }
  // values above the k-th are kept, and the first `left` (in index order) of those equal to it
  float best = -INFINITY;
  int arg = 0x7fffffff;
  if (tid == 0) s_taken = 0;
  __syncthreads();
  for (int base = 0; base < a.V; base += kSampleThreads) {
    const int i = base + tid;
    float v = 0.f;
    uint32_t o = 0;
    if (i < a.V) {
      v = (float)x[i];
      o = float_order(v);
    }
    const bool equal = i < a.V && o == prefix;
    const unsigned long long ballot = __builtin_amdgcn_ballot_w64(equal);
    if (lane == 0) s_wave[wave] = __builtin_popcountll(ballot);
    __syncthreads();
    int before = s_taken + __builtin_popcountll(ballot & ((1ull << lane) - 1));
    for (int w = 0; w < wave; ++w) before += s_wave[w];
    if (i < a.V && (o > prefix || (equal && before < left))) {
      const float z = a.u != nullptr ? with_noise(v, a.u[(int64_t)row * a.V + i], a.inv_temperature) : v;
      if (arg == 0x7fffffff || z > best || (z != z && best == best)) { best = z; arg = i; }
    }
    __syncthreads();
    if (tid == 0) {
      int n = 0;
      for (int w = 0; w < NW; ++w) n += s_wave[w];
      s_taken += n;
    }
    __syncthreads();
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const float ob = __shfl_xor(best, o);
    const int oa = __shfl_xor(arg, o);
    if (better_token(ob, oa, best, arg)) { best = ob; arg = oa; }
  }
  if (lane == 0) { s_best[wave] = best; s_arg[wave] = arg; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < NW; ++w)
      if (better_token(s_best[w], s_arg[w], best, arg)) { best = s_best[w]; arg = s_arg[w]; }
    a.out[(int64_t)row * a.out_ld] = arg;
    if (a.out2 != nullptr) a.out2[row] = arg;
  }
}

int launch_sample(const void* logits, int64_t ld, const float* u, int rows, int V, int k, float inv_temperature, int64_t* out, int64_t out_ld,
                  int64_t* out2, int dtype, hipStream_t stream) {
  const SampleArgs a = {logits, ld, u, V, k, inv_temperature, out, out_ld, out2};
  return by_type(dtype, true, [&](auto, auto t) {
    using T = decltype(t);
    if (V <= 256) hipLaunchKernelGGL((sample_few_kernel<T, 4>), dim3(rows), dim3(64), 0, stream, a);
    else if (V <= 512) hipLaunchKernelGGL((sample_few_kernel<T, 8>), dim3(rows), dim3(64), 0, stream, a);
    else hipLaunchKernelGGL((sample_kernel<T>), dim3(rows), dim3(kSampleThreads), 0, stream, a);
    return hipGetLastError() == hipSuccess ? 0 : -3;
  });
}

// y[m] = table[index[m]]: the embedding of one token per row.  One workgroup per row, 16 bytes per thread (the
// library's gather takes 9.7 us for 16 rows of 512, this a launch).  An index outside the table writes zeros.
__global__ __launch_bounds__(kThreads) void gather_rows_kernel(const char* table, int64_t row_bytes, int64_t ld_bytes, int64_t rows, const int64_t* index, char* y) {
  const int64_t i = index[blockIdx.x];
  for (int64_t o = 16 * threadIdx.x; o < row_bytes; o += 16 * kThreads) {
    vec<float, 4> v = {0.f, 0.f, 0.f, 0.f};
    if (i >= 0 && i < rows) v = *reinterpret_cast<const vec<float, 4>*>(table + i * ld_bytes + o);
    *reinterpret_cast<vec<float, 4>*>(y + blockIdx.x * row_bytes + o) = v;
  }
}
int launch_gather_rows(const void* table, int64_t row_bytes, int64_t ld_bytes, int64_t rows, const int64_t* index, int n, void* y, hipStream_t stream) {
  hipLaunchKernelGGL(gather_rows_kernel, dim3(n), dim3(kThreads), 0, stream, static_cast<const char*>(table), row_bytes, ld_bytes, rows, index,
                     static_cast<char*>(y));
  return hipGetLastError() == hipSuccess ? 0 : -3;
}

// ---------------------------------------------------------------------------
// Partial-result buffer of the entry point that allocates nothing: one array per GPU, part of the
// loaded code object, alive until the process ends.  Host code never uses the array's name as an
// address (on the host it is only a stand-in for the symbol): the device address is looked up
// once per device and handed to the kernels like any other workspace pointer.
static __device__ __align__(256) unsigned char scratch[kDecodeStaticScratchBytes];

int decode_static_scratch(float** ptr) {
  static std::mutex mu;
  static void* per_device[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return -3;
  std::lock_guard<std::mutex> lock(mu);
  if (per_device[dev] == nullptr) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || p == nullptr) return -3;
    per_device[dev] = p;
  }
  *ptr = static_cast<float*>(per_device[dev]);
  return 0;
}

// How many workgroups share the t rows of one (b, h).  Three workgroups a CU keep the memory busy (a
// fourth fits, and is not faster), so a launch runs in rounds of 3 CUs; a workgroup costs its iterations plus about two more for its start and end.  Fewest rounds x
// iterations wins, at least two iterations each.  45 x 6 heads of 450 rows: 26.1 us with the 2 splits this picks, 27.6
// with the 3 that fill a round and a straggling 5 % of the next; 16 x 8 heads of 540 rows: 16.6 us with one round,
// 20.7 with two.
int decode_pick_splits(int BH, int t, int rows_per_iteration, int cus) {
  if (t <= 0) return 1;
  const int64_t round = 3 * (int64_t)(cus > 0 ? cus : 256);
  const int most = std::min(64, (t + 2 * rows_per_iteration - 1) / (2 * rows_per_iteration));
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int s = 1; s <= most; ++s) {
    const int64_t iterations = ((t + s - 1) / s + rows_per_iteration - 1) / rows_per_iteration;
    const int64_t cost = ((int64_t)BH * s + round - 1) / round * (iterations + 2);
    if (cost < best_cost) { best_cost = cost; best = s; }
  }
  return best;
}

}  // namespace castle
