// Host side: from the run-time element type and head dimension of a call to template parameters.
#pragma once
#include <type_traits>
#include "castle_tiles.h"

namespace castle {

// f(compute type, tensor type): bf16 tensors are converted to fp16 on load (exact inside the fp16 range) and every
// operand produced inside the kernels is fp16, unless bf16_operands asks for bf16 MFMA operands
template <typename F> int by_type(int dtype, bool bf16_operands, F&& f) {
  switch (dtype) {
    case 0: return f(float(), float());
    case 1: return bf16_operands ? f(bf16_t(), bf16_t()) : f(fp16_t(), bf16_t());
    case 2: return f(fp16_t(), fp16_t());
    default: return -1;
  }
}
template <typename F> int by_type16(int dtype, bool bf16_operands, F&& f) {   // 16-bit tensors only
  if (dtype == 1) return bf16_operands ? f(bf16_t(), bf16_t()) : f(fp16_t(), bf16_t());
  return dtype == 2 ? f(fp16_t(), fp16_t()) : -1;
}
// f(std::integral_constant<int, d>); fp32 kernels exist up to d = 64
template <typename T, typename F> int by_head_dim(int d, F&& f) {
  switch (d) {
    case 16: return f(std::integral_constant<int, 16>());
    case 32: return f(std::integral_constant<int, 32>());
    case 64: return f(std::integral_constant<int, 64>());
    case 128:
      if constexpr (sizeof(T) == 2) return f(std::integral_constant<int, 128>());
      return -2;
    default: return -2;
  }
}

}  // namespace castle
