// Launcher of castle_gemm.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace castle {

enum { kGemmPlain = 0, kGemmGelu = 1, kGemmGeluSlope = 2 };
struct GemmArgs {
  const void *a, *b;   // contraction-contiguous: [free][ld], else [contraction][ld]
  void* c;             // [M][ldc]; a product that is split over the contraction needs ldc == N
  void* aux;           // kGemmGelu: gelu(c) goes here; kGemmGeluSlope: c is multiplied by the derivative of gelu at it; ldc rows
  int M, N, K;
  int64_t lda, ldb, ldc;
  int epilogue;
  int k_per_split;
  float* part;
  // largest |c| of the columns amax_from .. amax_to - 1 (a whole number of 16-byte pieces): one partial maximum per tile of them,
  // zeros in the other slots of the kAmaxBlocks at `amax`
  float* amax;
  int* amax_status;   // set to 0 if not nullptr
  int amax_from, amax_to;
  // rows of `a` are normalised on their way: a / sqrt(mean(a^2) + eps) * norm_w, kept in h (ld K) and their factors in rstd if not nullptr
  const void* norm_w;
  float eps;
  void* h;
  float* rstd;
};
// Weight gradient w (both operands contraction-strided) and input gradient x (the second one) of a projection in one launch: w_groups workgroups in rows of w_row,
// then x_groups in rows of x_row.
struct GradsArgs {
  GemmArgs w, x;
  int w_groups, w_row, x_groups, x_row;
};
constexpr int kNormBytes = 2048;   // longest row that a product normalises
bool gemm_norm_ok(int M, int N, int K, int elem_size);
bool gemm_amax_ok(int M, int N, int K, int elem_size, int amax_from, int amax_to);
void gemm_plan(int M, int N, int K, int elem_size, bool epilogue, int (&out)[4]);
int64_t gemm_workspace(int M, int N, int K, int elem_size, bool epilogue);
// fp32, castle_gemm32.hip
int launch_gemm32(const GemmArgs& a, bool a_kc, bool b_kc, int tile, int splits, int waves, hipStream_t stream);
int launch_grads32(const GradsArgs& p, int tile, int waves, hipStream_t stream);
struct GradsPlan { int tile, waves, w_splits, x_splits; };   // tile 0: two launches
GradsPlan grads_plan(int R, int N, int K, int elem_size, int epilogue, bool amax);
int64_t grads_workspace(int R, int N, int K, int elem_size, int epilogue, bool amax);   // -1: two launches are ahead
struct PartSum;
int launch_grads(GradsArgs p, int dtype, float* workspace, PartSum* later, hipStream_t stream);   // later: dw's sum is left to launch_sums, if it has one (parts > 0)
int launch_gemm(GemmArgs a, bool a_kc, bool b_kc, int dtype, float* workspace, hipStream_t stream);

}  // namespace castle
