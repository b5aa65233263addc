// Image front end of the vision encoders (vision.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace shai {
typedef uint16_t bf16_t;

// out [B (H / P) (W / P), P P 3] bf16: the pixels of every patch in the order (row, column, channel), normalised
// (u8 / 255 - mean) inv_std.  x [B, H, W, 3]; P % 8 == 0, H and W multiples of P, x 8-byte aligned.  With w, the weight of the
// convolution that they stand for, [w_pixels, 8] with channels of which three count, its [w_pixels, 3] goes to w_out: the product of
// the two needs no padded channels.  w_pixels % 4 == 0, both 16-byte aligned.
struct PatchArgs {
  const uint8_t* x;
  bf16_t* out;
  int B, H, W, P;
  float mean[3], inv_std[3];
  const bf16_t* w;
  bf16_t* w_out;
  long w_pixels;
};
[[nodiscard]] hipError_t launch_patches_u8(const PatchArgs& a, hipStream_t s);

// x [B, T, D] = (class token | patches | detection tokens) + position embedding, T = 1 + n + nd, and, where mr is given, mean and
// 1 / standard deviation [B T, 2] of its rows.  D % 8 == 0, D <= 2048.
struct TokenArgs {
  const bf16_t* patches;   // [B, n, D]
  const bf16_t* cls;       // [D]
  const bf16_t* det;       // [nd, D], nd > 0
  const bf16_t* pos;       // [T, D]
  bf16_t* out;
  float* mr;
  int B, n, nd, D;
  float eps;
};
[[nodiscard]] hipError_t launch_tokens(const TokenArgs& a, hipStream_t s);
}  // namespace shai
