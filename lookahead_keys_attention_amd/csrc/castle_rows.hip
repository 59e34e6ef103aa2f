// The per-row work between the products of a transformer block: RMS norm with the residual sum in front of it, its
// backward pass, mean cross entropy, the gradient of a token embedding, sums of partial weight gradients.
//
// All of it is bound by HBM: a few flops per element.  What the kernels save is passes.  A residual stream of 16384 x 512
// bf16 as operators of the tensor library: sum 9 us, norm 18, norm backward 35 + 17 + 5 for the weight, sum of the two
// gradients 9; here sum and norm together read two tensors and write two, and the backward pass reads three and writes
// one (figures at the kernels).  A row belongs to a group of 16, 32 or 64 lanes of one wave, so nothing crosses waves.
#include "castle_tiles.h"
#include "castle_rows.h"

namespace castle {
namespace {

constexpr int kRowWaves = kThreads / 64;

template <int LPR> __device__ __forceinline__ float row_sum(float v) {
#pragma unroll
  for (int o = 1; o < LPR; o <<= 1) v += __shfl_xor(v, o);
  return v;
}
template <int LPR> __device__ __forceinline__ float row_max(float v) {
#pragma unroll
  for (int o = 1; o < LPR; o <<= 1) v = fmaxf(v, __shfl_xor(v, o));
  return v;
}

// h = (x / sqrt(mean(x^2) + eps)) w with x = x0 + delta where a delta is given (the sum is rounded and stored like the
// operator would).  16384 x 512 bf16 with a sum: see castle_rows.h for the measured times.
template <typename T, int LPR, int NP> __global__ __launch_bounds__(kThreads) void norm_kernel(NormArgs a) {
  constexpr int V = elem_traits<T>::vec16, RPW = 64 / LPR;
  typedef vec<T, V> vt;
  typedef vec<float, V> vf;
  const int lane = lane_id(), sub = lane % LPR, pieces = a.D / V;
  const int64_t row = ((int64_t)blockIdx.x * kRowWaves + wave_id()) * RPW + lane / LPR;
  if (row >= a.rows) return;
  const int64_t at = row * a.D;
  vf x[NP], w[NP];
  float ssq = 0.f;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = p * LPR + sub;
#pragma unroll
    for (int e = 0; e < V; ++e) x[p][e] = w[p][e] = 0.f;
    if (i >= pieces) continue;
    x[p] = __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.x) + at + i * V), vf);
    w[p] = __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.w) + i * V), vf);
    if (a.delta != nullptr) {
      x[p] += __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.delta) + at + i * V), vf);
      const vt r = __builtin_convertvector(x[p], vt);
      *reinterpret_cast<vt*>(static_cast<T*>(a.sum) + at + i * V) = r;
      x[p] = __builtin_convertvector(r, vf);
    }
  }
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int e = 0; e < V; ++e) ssq = __builtin_fmaf(x[p][e], x[p][e], ssq);
  const float r = 1.f / sqrtf(row_sum<LPR>(ssq) / (float)a.D + a.eps);
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = p * LPR + sub;
    if (i < pieces) *reinterpret_cast<vt*>(static_cast<T*>(a.h) + at + i * V) = __builtin_convertvector(x[p] * r * w[p], vt);
  }
  if (sub == 0 && a.rstd != nullptr) a.rstd[row] = r;
}

// dx = dres + r (w dh - xr mean(w dh xr)) with xr = x r; partial sums of dw = sum over rows of dh xr, one row of
// dw_part per workgroup.  16384 x 512 bf16 with dres: 13.7 us + 5.2 for the column sums (67 us as four operators).
template <typename T, int LPR, int NP> __global__ __launch_bounds__(kThreads) void norm_bwd_kernel(NormBwdArgs a) {
  constexpr int V = elem_traits<T>::vec16, RPW = 64 / LPR;
  typedef vec<T, V> vt;
  typedef vec<float, V> vf;
  extern __shared__ float s_dw[];   // [D]
  const int lane = lane_id(), wave = wave_id(), sub = lane % LPR, pieces = a.D / V;
  const int64_t step = (int64_t)gridDim.x * kRowWaves * RPW;
  vf w[NP], dw[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int i = p * LPR + sub;
#pragma unroll
    for (int e = 0; e < V; ++e) w[p][e] = dw[p][e] = 0.f;
    if (i < pieces) w[p] = __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.w) + i * V), vf);
  }
  for (int64_t row = ((int64_t)blockIdx.x * kRowWaves + wave) * RPW + lane / LPR; row < a.rows; row += step) {
    const int64_t at = row * a.D;
    vf x[NP], d[NP], res[NP];
    const float r = a.rstd[row];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int i = p * LPR + sub;
#pragma unroll
      for (int e = 0; e < V; ++e) x[p][e] = d[p][e] = res[p][e] = 0.f;
      if (i >= pieces) continue;
      x[p] = __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.x) + at + i * V), vf);
      d[p] = __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.dh) + at + i * V), vf);
      if (a.dres != nullptr) res[p] = __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.dres) + at + i * V), vf);
    }
    float dot = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int e = 0; e < V; ++e) {
        x[p][e] *= r;
        dw[p][e] = __builtin_fmaf(d[p][e], x[p][e], dw[p][e]);
        d[p][e] *= w[p][e];
        dot = __builtin_fmaf(d[p][e], x[p][e], dot);
      }
    const float m = row_sum<LPR>(dot) / (float)a.D;
    if (a.dx != nullptr) {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int i = p * LPR + sub;
        if (i < pieces)
          *reinterpret_cast<vt*>(static_cast<T*>(a.dx) + at + i * V) = __builtin_convertvector(res[p] + (d[p] - x[p] * m) * r, vt);
      }
    }
  }
  if (a.dw_part == nullptr) return;
#pragma unroll
  for (int p = 0; p < NP; ++p)
#pragma unroll
    for (int e = 0; e < V; ++e)
#pragma unroll
      for (int o = LPR; o < 64; o <<= 1) dw[p][e] += __shfl_xor(dw[p][e], o);
  for (int t = 0; t < kRowWaves; ++t) {
    if (wave == t && lane < LPR) {
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const int i = p * LPR + sub;
        if (i < pieces)
#pragma unroll
          for (int e = 0; e < V; ++e) s_dw[i * V + e] = (t ? s_dw[i * V + e] : 0.f) + dw[p][e];
      }
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < a.D; i += kThreads) a.dw_part[(int64_t)blockIdx.x * a.D + i] = s_dw[i];
}

// out[i] = sum over the G rows of part[G][D]: 16 columns of a workgroup, 16 threads down each of them
template <typename T> __device__ __forceinline__ void column_sum(const float* part, int G, int D, T* out, int block) {
  __shared__ float s[16][17];
  const int c = threadIdx.x % 16, r = threadIdx.x / 16, col = block * 16 + c;
  float v = 0.f;
  if (col < D) {
#pragma unroll 8
    for (int g = r; g < G; g += 16) v += part[(int64_t)g * D + col];
  }
  s[r][c] = v;
  __syncthreads();
  if (r == 0 && col < D) {
#pragma unroll
    for (int k = 1; k < 16; ++k) v += s[k][c];
    out[col] = (T)v;
  }
}

// out[i] = sum over P of part[P][n], n a multiple of 8: the partial products of a weight gradient.  8 parts of 512 x 512 ...
// 3072 x 512: 6.7 us on average, 14 as a sum and a conversion of their own.
template <typename T> __device__ __forceinline__ void part_sum(const float* part, int P, int64_t n, T* out, int block) {
  const int64_t i = ((int64_t)block * kThreads + threadIdx.x) * 8;
  if (i >= n) return;
  typedef vec<float, 4> v4;
  v4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll 8
  for (int p = 0; p < P; ++p) {
    a += *reinterpret_cast<const v4*>(part + p * n + i);
    b += *reinterpret_cast<const v4*>(part + p * n + i + 4);
  }
  vec<float, 8> s;
#pragma unroll
  for (int e = 0; e < 4; ++e) { s[e] = a[e]; s[4 + e] = b[e]; }
  *reinterpret_cast<frag_mem<T>*>(out + i) = __builtin_convertvector(s, frag<T>);
}

// Several sums, each of the workgroups first[j] .. first[j + 1] - 1.  A sum by itself is a launch of 4 us for 1 to 3 MB, hardly more than its start.
template <typename T> __global__ __launch_bounds__(kThreads) void sums_kernel(SumsArgs a) {
  PartSum job = a.job[0];
  int block = blockIdx.x;
#pragma unroll
  for (int j = 1; j < kMaxSums; ++j)
    if ((int)blockIdx.x >= a.first[j]) {
      job = a.job[j];
      block = blockIdx.x - a.first[j];
    }
  if (job.columns) column_sum<T>(job.part, job.parts, (int)job.n, static_cast<T*>(job.out), block);
  else part_sum<T>(job.part, job.parts, job.n, static_cast<T*>(job.out), block);
}

// Mean cross entropy of rows of logits against class numbers (torch's default ignore_index -100 does not count; a class
// outside 0 .. V - 1 makes the loss and its row's gradient NaN).  One wave per row; lse of every row is kept for the backward pass.  16384 x 256
// bf16 in the layout the logits come in: under 10 us each way (190 and 176 us as operators on the transposed logits).
__device__ __forceinline__ int64_t target_of(const CrossEntropyArgs& a, int64_t row) { return a.target[row / a.n * a.target_ld + row % a.n]; }

template <typename T> __global__ __launch_bounds__(kThreads) void ce_kernel(CrossEntropyArgs a) {
  constexpr int V = elem_traits<T>::vec16;
  typedef vec<T, V> vt;
  typedef vec<float, V> vf;
  __shared__ float s_sum[kRowWaves], s_cnt[kRowWaves];
  const int lane = lane_id(), wave = wave_id(), pieces = a.V / V;
  float sum = 0.f, cnt = 0.f;
  for (int64_t row = (int64_t)blockIdx.x * kRowWaves + wave; row < a.rows; row += (int64_t)gridDim.x * kRowWaves) {
    const T* x = static_cast<const T*>(a.logits) + row * a.V;
    const int64_t t = target_of(a, row);
    float m = -INFINITY, s = 0.f;
    for (int i = lane; i < pieces; i += 64) {
      const vf v = __builtin_convertvector(*reinterpret_cast<const vt*>(x + i * V), vf);
      float mn = m;
#pragma unroll
      for (int e = 0; e < V; ++e) mn = fmaxf(mn, v[e]);
      s *= m == -INFINITY ? 0.f : fast_exp2((m - mn) * kLog2e);
#pragma unroll
      for (int e = 0; e < V; ++e) s += mn == -INFINITY ? v[e] != v[e] ? NAN : 0.f : fast_exp2((v[e] - mn) * kLog2e);   // (fmaxf drops NaNs)
      m = mn;
    }
    const float M = row_max<64>(m);
    const float lse = M + logf(row_sum<64>(m == -INFINITY ? s : s * fast_exp2((m - M) * kLog2e)));   // (nothing seen but -inf: 0, or NaN)
    if (lane == 0) a.lse[row] = lse;
    if (t == -100) continue;
    sum += t >= 0 && t < a.V ? lse - (float)x[t] : NAN;
    cnt += 1.f;
  }
  if (lane == 0) { s_sum[wave] = sum; s_cnt[wave] = cnt; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kRowWaves; ++k) { sum += s_sum[k]; cnt += s_cnt[k]; }
    a.part[2 * blockIdx.x] = sum;
    a.part[2 * blockIdx.x + 1] = cnt;
  }
}
// the mean over G partial sums; 1 / count is kept for the backward pass
template <typename T> __global__ __launch_bounds__(kThreads) void ce_mean_kernel(const float* part, int G, T* loss, float* inv_count) {
  __shared__ float s_sum[kRowWaves], s_cnt[kRowWaves];
  float sum = 0.f, cnt = 0.f;
  for (int i = threadIdx.x; i < G; i += kThreads) { sum += part[2 * i]; cnt += part[2 * i + 1]; }
  sum = row_sum<64>(sum);
  cnt = row_sum<64>(cnt);
  if (lane_id() == 0) { s_sum[wave_id()] = sum; s_cnt[wave_id()] = cnt; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int k = 1; k < kRowWaves; ++k) { sum += s_sum[k]; cnt += s_cnt[k]; }
    *loss = (T)(sum / cnt);
    *inv_count = 1.f / cnt;
  }
}
template <typename T> __global__ __launch_bounds__(kThreads) void ce_bwd_kernel(CrossEntropyArgs a, const T* grad, const float* inv_count, T* dlogits) {
  constexpr int V = elem_traits<T>::vec16;
  typedef vec<T, V> vt;
  typedef vec<float, V> vf;
  const int lane = lane_id(), pieces = a.V / V;
  const int64_t row = (int64_t)blockIdx.x * kRowWaves + wave_id();
  if (row >= a.rows) return;
  const int64_t t = target_of(a, row), at = row * a.V;
  const bool counts = t != -100;
  const float g = t >= 0 && t < a.V ? (float)*grad * *inv_count : NAN, lse = a.lse[row];
  for (int i = lane; i < pieces; i += 64) {
    const vf v = __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.logits) + at + i * V), vf);
    vf d;
#pragma unroll
    for (int e = 0; e < V; ++e) d[e] = !counts ? 0.f : g * (fast_exp2((v[e] - lse) * kLog2e) - (t == i * V + e ? 1.f : 0.f));
    *reinterpret_cast<vt*>(dlogits + at + i * V) = __builtin_convertvector(d, vt);
  }
}

// Gradient of an embedding: part[c][v] = sum of the dy rows of chunk c whose token is v.  A workgroup takes one
// vocabulary row and one chunk of at most kChunk tokens, lists the matches in order and adds their rows: no sort, no atomics, the
// same sum every time (16384 tokens of 256 x 512: 14 us; a sort, its scans and a wait of the host as an operator).  Every workgroup reads its chunk's token numbers, so this is for small vocabularies (the
// rule is the caller's: castle_embedding_grad).
constexpr int kChunk = 2048;
template <typename T> __global__ __launch_bounds__(kThreads) void embedding_grad_kernel(EmbeddingGradArgs a) {
  constexpr int V = elem_traits<T>::vec16;
  typedef vec<T, V> vt;
  typedef vec<float, V> vf;
  __shared__ int s_list[kChunk], s_wave[kRowWaves];
  extern __shared__ float s_row[];   // [D]
  const int lane = lane_id(), wave = wave_id(), v = blockIdx.x, pieces = a.D / V;
  const int64_t r0 = (int64_t)blockIdx.y * kChunk, r1 = r0 + kChunk < a.rows ? r0 + kChunk : a.rows;
  int found = 0;
  for (int64_t base = r0; base < r1; base += kThreads) {
    const int64_t r = base + threadIdx.x;
    const bool hit = r < r1 && a.index[r / a.n * a.index_ld + r % a.n] == v;
    const uint64_t mask = __ballot(hit);
    if (lane == 0) s_wave[wave] = __popcll(mask);
    __syncthreads();
    int before = found, all = 0;
#pragma unroll
    for (int k = 0; k < kRowWaves; ++k) {
      before += k < wave ? s_wave[k] : 0;
      all += s_wave[k];
    }
    if (hit) s_list[before + __popcll(mask & ((1ull << lane) - 1))] = (int)(r - r0);
    found += all;
    __syncthreads();
  }
  // a wave takes every fourth match; pieces of a row go over its lanes
  for (int p0 = 0; p0 < pieces; p0 += 64) {
    const int i = p0 + lane;
    vf acc;
#pragma unroll
    for (int e = 0; e < V; ++e) acc[e] = 0.f;
    if (i < pieces) {
#pragma unroll 4
      for (int k = wave; k < found; k += kRowWaves)
        acc += __builtin_convertvector(*reinterpret_cast<const vt*>(static_cast<const T*>(a.dy) + (r0 + s_list[k]) * a.D + i * V), vf);
    }
    for (int t = 0; t < kRowWaves; ++t) {
      if (wave == t && i < pieces)
#pragma unroll
        for (int e = 0; e < V; ++e) s_row[i * V + e] = (t ? s_row[i * V + e] : 0.f) + acc[e];
      __syncthreads();
    }
  }
  float* out = a.part + ((int64_t)blockIdx.y * a.V + v) * a.D;
  for (int i = threadIdx.x; i < a.D; i += kThreads) out[i] = s_row[i];
}

// f(std::integral_constant lanes of a row, std::integral_constant pieces of a lane) for rows of `pieces` 16-byte pieces
template <typename F> int by_row_length(int pieces, F&& f) {
  using std::integral_constant;
  if (pieces <= 16) return f(integral_constant<int, 16>(), integral_constant<int, 1>());
  if (pieces <= 32) return f(integral_constant<int, 32>(), integral_constant<int, 1>());
  if (pieces <= 64) return f(integral_constant<int, 64>(), integral_constant<int, 1>());
  if (pieces <= 128) return f(integral_constant<int, 64>(), integral_constant<int, 2>());
  if (pieces <= 256) return f(integral_constant<int, 64>(), integral_constant<int, 4>());
  if (pieces <= kMaxRowPieces) return f(integral_constant<int, 64>(), integral_constant<int, 8>());
  return -2;
}
template <typename F> int by_tensor_type(int dtype, F&& f) {
  switch (dtype) {
    case 0: return f(float());
    case 1: return f(bf16_t());
    case 2: return f(fp16_t());
    default: return -1;
  }
}
int launched() { return hipGetLastError() == hipSuccess ? 0 : -3; }

}  // namespace

int launch_norm(const NormArgs& a, int dtype, hipStream_t stream) {
  return by_tensor_type(dtype, [&](auto t) {
    using T = decltype(t);
    return by_row_length(a.D / elem_traits<T>::vec16, [&](auto lpr, auto np) {
      constexpr int rows = kRowWaves * (64 / lpr.value);
      hipLaunchKernelGGL((norm_kernel<T, lpr.value, np.value>), dim3((unsigned)((a.rows + rows - 1) / rows)), dim3(kThreads), 0, stream, a);
      return launched();
    });
  });
}

// two rounds of a resident workgroup's rows at most leave a CU idle, and more partial rows cost the second launch time
int norm_bwd_groups(int64_t rows, int D, int elem_size) {
  const int pieces = D * elem_size / 16, per = kRowWaves * (pieces <= 16 ? 4 : pieces <= 32 ? 2 : 1);
  const int64_t g = (rows + 2 * per - 1) / (2 * per);
  return (int)(g < 1 ? 1 : g > 1024 ? 1024 : g);
}

int launch_norm_bwd(const NormBwdArgs& a, void* dw, int dtype, PartSum* later, hipStream_t stream) {
  return by_tensor_type(dtype, [&](auto t) {
    using T = decltype(t);
    const int groups = norm_bwd_groups(a.rows, a.D, (int)sizeof(T));
    const int rc = by_row_length(a.D / elem_traits<T>::vec16, [&](auto lpr, auto np) {
      hipLaunchKernelGGL((norm_bwd_kernel<T, lpr.value, np.value>), dim3(groups), dim3(kThreads), a.D * sizeof(float), stream, a);
      return launched();
    });
    if (rc != 0 || a.dw_part == nullptr) return rc;
    const PartSum sum = {a.dw_part, a.D, dw, groups, 1};
    if (later != nullptr) *later = sum;
    return later != nullptr ? 0 : launch_sums(&sum, 1, dtype, stream);
  });
}

int launch_sums(const PartSum* sums, int count, int dtype, hipStream_t stream) {
  SumsArgs a = {};
  int64_t blocks = 0;
  for (int j = 0; j < kMaxSums; ++j) {
    a.first[j] = j < count ? (int)blocks : 0x7fffffff;
    if (j >= count) continue;
    a.job[j] = sums[j];
    const int64_t per = sums[j].columns ? 16 : 8 * kThreads;
    blocks += (sums[j].n + per - 1) / per;
    if (blocks > 0x7ffffff0) return -2;
  }
  return by_tensor_type(dtype, [&](auto t) {
    hipLaunchKernelGGL((sums_kernel<decltype(t)>), dim3((unsigned)blocks), dim3(kThreads), 0, stream, a);
    return launched();
  });
}
int launch_part_sum(const float* part, int parts, int64_t n, void* out, int dtype, hipStream_t stream) {
  const PartSum sum = {part, n, out, parts, 0};
  return launch_sums(&sum, 1, dtype, stream);
}

int cross_entropy_groups(int64_t rows) {
  const int64_t g = (rows + kRowWaves - 1) / kRowWaves;
  return (int)(g > kCrossEntropyGroups ? kCrossEntropyGroups : g);
}
int launch_cross_entropy(const CrossEntropyArgs& a, void* loss, float* inv_count, int dtype, hipStream_t stream) {
  return by_tensor_type(dtype, [&](auto t) {
    using T = decltype(t);
    const int groups = cross_entropy_groups(a.rows);
    hipLaunchKernelGGL((ce_kernel<T>), dim3(groups), dim3(kThreads), 0, stream, a);
    hipLaunchKernelGGL((ce_mean_kernel<T>), dim3(1), dim3(kThreads), 0, stream, a.part, groups, static_cast<T*>(loss), inv_count);
    return launched();
  });
}
int launch_cross_entropy_bwd(const CrossEntropyArgs& a, const void* grad, const float* inv_count, void* dlogits, int dtype, hipStream_t stream) {
  return by_tensor_type(dtype, [&](auto t) {
    using T = decltype(t);
    hipLaunchKernelGGL((ce_bwd_kernel<T>), dim3((unsigned)((a.rows + kRowWaves - 1) / kRowWaves)), dim3(kThreads), 0, stream, a, static_cast<const T*>(grad),
                       inv_count, static_cast<T*>(dlogits));
    return launched();
  });
}

int embedding_grad_chunks(int64_t rows) { return (int)((rows + kChunk - 1) / kChunk); }
int launch_embedding_grad(const EmbeddingGradArgs& a, void* dw, int dtype, hipStream_t stream) {
  return by_tensor_type(dtype, [&](auto t) {
    using T = decltype(t);
    const int chunks = embedding_grad_chunks(a.rows);
    hipLaunchKernelGGL((embedding_grad_kernel<T>), dim3(a.V, chunks), dim3(kThreads), a.D * sizeof(float), stream, a);
    if (launched() != 0) return -3;
    return launch_part_sum(a.part, chunks, (int64_t)a.V * a.D, dw, dtype, stream);
  });
}

}  // namespace castle
