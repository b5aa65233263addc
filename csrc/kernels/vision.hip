// Image front end of the vision encoders: what stands before the first layer, in two launches beside the patch product.
//
// Bytes bound both at a batch (32 images of 224 x 224: 4.8 MB in and 9.6 out, 9.6 in and 9.7 out), launches at one image.  Before,
// a cast, two affine passes, a cast, the channels' padding from 3 to 8 (which also made the patch product 2048 deep instead of 768),
// a concatenation, a copy, an addition and the row moments were launches of their own.
#include "common.h"
#include "launch.h"
#include "vision.h"

namespace shai {

// A thread takes 8 adjacent bytes of a patch's row: 16 bytes out.  Workgroups from image_blocks on take the weight, 4 pixels a thread: on
// every call, so that the product reads the parameter as it is then, also in a replay of a graph.  The weight's 3.1 MB are read by CUs
// that one image's 74 workgroups leave idle: a pass of ViT-base with a weight stripped beforehand 570 us, so 571
// (this launch 3.5 us, 7.1 for 32 images).
__global__ void __launch_bounds__(256) patches_u8_kernel(const PatchArgs a, long total, unsigned image_blocks) {
  if (blockIdx.x >= image_blocks) {
    const long j = (blockIdx.x - image_blocks) * 256L + threadIdx.x;
    if (j * 4 >= a.w_pixels) return;
    uint2_ v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const uint2_*>(a.w + (j * 4 + e) * 8);
    uint2_* out = reinterpret_cast<uint2_*>(a.w_out + j * 12);
    out[0] = uint2_{v[0][0], (v[0][1] & 0xffffu) | v[1][0] << 16};
    out[1] = uint2_{v[1][0] >> 16 | v[1][1] << 16, v[2][0]};
    out[2] = uint2_{(v[2][1] & 0xffffu) | v[3][0] << 16, v[3][0] >> 16 | v[3][1] << 16};
    return;
  }
  const long i = blockIdx.x * 256L + threadIdx.x;
  if (i >= total) return;
  const int per_row = a.P * 3 / 8;                     // 8-byte pieces of a patch's row
  const int gw = a.W / a.P;
  const int piece = (int)(i % per_row);
  long r = i / per_row;
  const int ky = (int)(r % a.P);
  r /= a.P;                                            // patch
  const int gx = (int)(r % gw);
  const long y = r / gw * a.P + ky;                    // image rows lie one after the other: b H + gy P + ky
  const uint2_ v = *reinterpret_cast<const uint2_*>(a.x + (y * a.W + (long)gx * a.P) * 3 + piece * 8);
  float f[8];
  int c = piece * 8 % 3;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float u = __fmul_rn((float)((v[e >> 2] >> (8 * (e & 3))) & 255u), 1.f / 255.f);
    const float mean = c == 0 ? a.mean[0] : c == 1 ? a.mean[1] : a.mean[2];
    const float inv = c == 0 ? a.inv_std[0] : c == 1 ? a.inv_std[1] : a.inv_std[2];
    f[e] = __fmul_rn(__fsub_rn(u, mean), inv);
    c = c == 2 ? 0 : c + 1;
  }
  *reinterpret_cast<uint4_*>(a.out + i * 8) = pack8(f);
}

hipError_t launch_patches_u8(const PatchArgs& a, hipStream_t s) {
  const long total = (long)a.B * a.H * a.W * 3 / 8;
  const unsigned images = (unsigned)((total + 255) / 256), weight = a.w ? (unsigned)((a.w_pixels / 4 + 255) / 256) : 0;
  return images + weight > 0 ? launch(patches_u8_kernel, images + weight, 256, s, a, total, images) : hipSuccess;
}

// One wave a row, held in registers; mean and variance in two passes over them.
template <int V>
__global__ void __launch_bounds__(256) tokens_kernel(const TokenArgs a) {
  const int lane = threadIdx.x & 63, T = 1 + a.n + a.nd;
  const long row = blockIdx.x * 4L + (threadIdx.x >> 6);
  if (row >= (long)a.B * T) return;
  const long b = row / T;
  const int t = (int)(row - b * T);
  const bf16_t* src = t == 0 ? a.cls : t <= a.n ? a.patches + (b * a.n + t - 1) * a.D : a.det + (long)(t - 1 - a.n) * a.D;
  const bf16_t* pos = a.pos + (long)t * a.D;
  uint4_ v[V];
  float sum = 0.f;
#pragma unroll
  for (int c = 0; c < V; ++c) {
    const int col = (c * 64 + lane) * 8;
    v[c] = uint4_{0, 0, 0, 0};
    if (col < a.D) {
      float f[8], p[8];
      unpack8(*reinterpret_cast<const uint4_*>(src + col), f);
      unpack8(*reinterpret_cast<const uint4_*>(pos + col), p);
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] += p[e];
      v[c] = pack8(f);
      *reinterpret_cast<uint4_*>(a.out + row * a.D + col) = v[c];
      unpack8(v[c], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += f[e];
    }
  }
  if (a.mr == nullptr) return;
  const float mean = wave_sum(sum) / a.D;
  float var = 0.f;
#pragma unroll
  for (int c = 0; c < V; ++c) {
    if ((c * 64 + lane) * 8 >= a.D) continue;
    float f[8];
    unpack8(v[c], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) var = fmaf(f[e] - mean, f[e] - mean, var);
  }
  var = wave_sum(var) / a.D;
  if (lane == 0) *reinterpret_cast<float2*>(a.mr + 2 * row) = make_float2(mean, rsqrtf(var + a.eps));
}

hipError_t launch_tokens(const TokenArgs& a, hipStream_t s) {
  const long rows = (long)a.B * (1 + a.n + a.nd);
  if (rows <= 0) return hipSuccess;
  const unsigned grid = (unsigned)((rows + 3) / 4);
  return launch(a.D <= 512 ? tokens_kernel<1> : a.D <= 1024 ? tokens_kernel<2> : tokens_kernel<4>, grid, 256, s, a);
}

}  // namespace shai
