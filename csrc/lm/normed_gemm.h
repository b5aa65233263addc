// The residual's norm in the product that reads it (normed_gemm.hip).
#pragma once
#include "lm.h"

namespace shai_lm {

struct NormedGemmArgs {
  const float* x;          // [M, K] residual, or null: x = table[ids] * scale
  const int* ids;
  const void* table;       // [V, K] bf16
  float scale;
  int V;
  const float* delta;      // [parts, M, K] partial sums of a sublayer's output, added to x; or null
  int parts;
  long part_stride;
  const float* w;          // [K] gain
  float eps;
  int width;               // K before padding
  float* x_out;            // [M, K] x + delta, apart from x; or null
  GemmArgs g;              // A: the norm of x_out in bf16
};
bool normed_gemm_fits(int M, int K, int parts);
void launch_normed_gemm(const NormedGemmArgs& a, hipStream_t s);       // plain and squared-ReLU epilogues

}  // namespace shai_lm
