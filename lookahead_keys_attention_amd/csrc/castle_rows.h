// Launchers of castle_rows.hip: rows of D (or V) elements, contiguous, a whole number of 16-byte pieces.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace castle {

constexpr int kMaxRowPieces = 512;        // 16-byte pieces of a row that the norm kernels hold in registers
constexpr int kCrossEntropyGroups = 1024; // partial sums of the loss

struct NormArgs {
  const void *x, *delta;   // delta: nullptr, or a tensor added to x first; the sum goes to `sum`
  const void* w;
  void *sum, *h;
  float* rstd;             // 1 / rms of every row for the backward pass, or nullptr
  int64_t rows;
  int D;
  float eps;
};
int launch_norm(const NormArgs& a, int dtype, hipStream_t stream);

struct NormBwdArgs {
  const void *dh, *x, *w, *dres;   // dres: nullptr, or a gradient added to dx
  const float* rstd;
  void* dx;                        // nullptr: only the weight's gradient
  float* dw_part;                  // [norm_bwd_groups][D], or nullptr when the weight's gradient is not wanted
  int64_t rows;
  int D;
};
int norm_bwd_groups(int64_t rows, int D, int elem_size);
// out[n] = sum over `parts` rows of part[parts][n]: eight columns a thread (n a multiple of 8), or with `columns` sixteen threads down a column of few
struct PartSum {
  const float* part;
  int64_t n;
  void* out;
  int32_t parts, columns;
};
constexpr int kMaxSums = 4;
struct SumsArgs {
  PartSum job[kMaxSums];
  int first[kMaxSums];   // workgroup
};
int launch_sums(const PartSum* sums, int count, int dtype, hipStream_t stream);
// later: the sum of the weight's gradient is left to launch_sums
int launch_norm_bwd(const NormBwdArgs& a, void* dw, int dtype, PartSum* later, hipStream_t stream);

int launch_part_sum(const float* part, int parts, int64_t n, void* out, int dtype, hipStream_t stream);

struct CrossEntropyArgs {
  const void* logits;      // [rows][V]
  const int64_t* target;   // row r: target[(r / n) * target_ld + r % n]
  int64_t rows, n, target_ld;
  int V;
  float* lse;              // [rows]
  float* part;             // [cross_entropy_groups][2]
};
int cross_entropy_groups(int64_t rows);
int launch_cross_entropy(const CrossEntropyArgs& a, void* loss, float* inv_count, int dtype, hipStream_t stream);
int launch_cross_entropy_bwd(const CrossEntropyArgs& a, const void* grad, const float* inv_count, void* dlogits, int dtype, hipStream_t stream);

struct EmbeddingGradArgs {
  const void* dy;          // [rows][D]
  const int64_t* index;    // like CrossEntropyArgs::target
  int64_t rows, n, index_ld;
  int V, D;
  float* part;             // [embedding_grad_chunks][V][D]
};
int embedding_grad_chunks(int64_t rows);
int launch_embedding_grad(const EmbeddingGradArgs& a, void* dw, int dtype, hipStream_t stream);

}  // namespace castle
