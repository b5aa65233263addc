// The fold of a split-K product with the row norm that reads it (fold_norm.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace shai {
typedef uint16_t bf16_t;

// y = sum of the parts + bias + res_alpha residual; out = RMS norm or LayerNorm of y as stored.
struct FoldNormArgs {
  const float* parts;      // [splits, rows, D]
  const bf16_t* bias;      // [D] or null
  const bf16_t* residual;  // [rows, D] with row stride ldr, or null
  bf16_t* y;               // [rows, D]
  const bf16_t* gamma;     // [D] or null
  const bf16_t* beta;      // [D] or null
  bf16_t* out;             // [rows, D]
  int splits, rows, D, rms;
  long ldr;
  float res_alpha, eps;
};
// D a multiple of 4 up to 2048, every address and ldr of 8 bytes
bool fold_norm_supported(const FoldNormArgs& a);
[[nodiscard]] hipError_t launch_fold_norm(const FoldNormArgs& a, hipStream_t s);
}  // namespace shai
