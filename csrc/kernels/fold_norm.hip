// Fold of split-K partial sums, residual and the next row norm in one launch.
//
// A layer of a small batch is a chain of launches that cost 3.5 to 4.5 us each whatever they do: a product whose K is split over
// workgroups, its fold, the norm of the result, the next product.  The fold and the norm read some hundred KB: all loads of a row are
// issued before the first addition, by a wave for every 256 columns, and the row never leaves the registers between the two.
// us apart -> one launch: 154 x 1024 x 4096 13.9 -> 10.5, 197 x 768 x 3072 13.5 -> 9.9, 512 x 1280 x 5120 25.2 -> 21.3; where K was not split
// before, splitting it pays now: 197 x 768 x 768 8.6 -> 7.6.  A row a wave, its parts four at a time, took 0.3 to 1.2 us longer: 32 x 1024 x
// 2816 in 8 parts 9.0 -> 7.8, 128 x 1280 x 1280 in 2 9.7 -> 9.1, 197 x 768 x 3072 in 4 10.1 -> 9.8.
#include "fold_norm.h"
#include "common.h"
#include "launch.h"

namespace shai {

namespace {

__device__ __forceinline__ float at4(const uint2_& t, int e) { return bf2f(e & 1 ? t[e >> 1] >> 16 : t[e >> 1] & 0xffff); }

__device__ __forceinline__ uint2_ pack4(const float (&f)[4]) { return uint2_{pack2(f[0], f[1]), pack2(f[2], f[3])}; }

// W: waves, each 256 columns of the row, 4 a lane.  The parts are added in the order, and the bias and the residual with the operations, of
// gemm_splitk_reduce: y has the bits that it writes.
template <int W>
__global__ void __launch_bounds__(64 * W) fold_norm_kernel(const FoldNormArgs p) {
  constexpr int ROUND = 16;   // parts in flight
  __shared__ float red[2][W];
  const int tid = threadIdx.x;
  const long row = blockIdx.x, slab = (long)p.rows * p.D;
  const bool in = tid * 4 < p.D;
  const int col = in ? tid * 4 : 0;   // spare lanes read column 0
  const float* src = p.parts + row * p.D + col;
  auto load = [&](const bf16_t* at) { return *reinterpret_cast<const uint2_*>(at + col); };
  const uint2_ one = {0x3f803f80u, 0x3f803f80u}, zero = {0u, 0u};
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  uint2_ r, bias, gain, shift;
  for (int s0 = 0; s0 < p.splits; s0 += ROUND) {
    float4_ x[ROUND];
#pragma unroll
    for (int u = 0; u < ROUND; ++u)
      if (s0 + u < p.splits) x[u] = *reinterpret_cast<const float4_*>(src + (s0 + u) * slab);
    if (s0 == 0) {
      r = p.residual ? load(p.residual + row * p.ldr) : zero;
      bias = p.bias ? load(p.bias) : zero;
      gain = p.gamma ? load(p.gamma) : one;
      shift = p.beta ? load(p.beta) : zero;
    }
#pragma unroll
    for (int u = 0; u < ROUND; ++u)
      if (s0 + u < p.splits) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += x[u][e];
      }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (p.bias) v[e] += at4(bias, e);
    if (p.residual) v[e] += at4(r, e) * p.res_alpha;
  }
  const uint2_ w = pack4(v);
  if (in) *reinterpret_cast<uint2_*>(p.y + row * p.D + col) = w;
  float sum = 0.f, sq = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = in ? at4(w, e) : 0.f;   // as the next layer reads it
    sum += v[e];
    sq += v[e] * v[e];
  }
  auto total = [&](float t, float* at) {   // over the row
    t = wave_sum(t);
    if constexpr (W == 1) return t;
    if ((tid & 63) == 0) at[tid >> 6] = t;
    __syncthreads();
    t = at[0];
#pragma unroll
    for (int u = 1; u < W; ++u) t += at[u];
    return t;
  };
  float mean = 0.f, rstd;
  if (p.rms) {
    rstd = rsqrtf(total(sq, red[0]) / p.D + p.eps);
  } else {
    mean = total(sum, red[0]) / p.D;
    float var = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = in ? v[e] - mean : 0.f;
      var += d * d;
    }
    rstd = rsqrtf(total(var, red[1]) / p.D + p.eps);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = (v[e] - mean) * rstd * at4(gain, e) + at4(shift, e);
  if (in) *reinterpret_cast<uint2_*>(p.out + row * p.D + col) = pack4(v);
}

}  // namespace

bool fold_norm_supported(const FoldNormArgs& a) {
  const uintptr_t at = (uintptr_t)a.bias | (uintptr_t)a.residual | (uintptr_t)a.y | (uintptr_t)a.gamma | (uintptr_t)a.beta | (uintptr_t)a.out;
  return a.D % 4 == 0 && a.D <= 2048 && (at & 7) == 0 && (a.residual == nullptr || a.ldr % 4 == 0);
}

hipError_t launch_fold_norm(const FoldNormArgs& a, hipStream_t s) {
  if (a.rows == 0) return hipSuccess;
  if (!fold_norm_supported(a)) return hipErrorInvalidValue;
  const int waves = (a.D + 255) / 256;
  auto go = [&](auto kernel, int w) { return launch(kernel, a.rows, 64 * w, s, a); };
  return waves <= 1 ? go(fold_norm_kernel<1>, 1) : waves <= 2 ? go(fold_norm_kernel<2>, 2) : waves <= 3 ? go(fold_norm_kernel<3>, 3)
         : waves <= 4 ? go(fold_norm_kernel<4>, 4) : waves <= 5 ? go(fold_norm_kernel<5>, 5) : go(fold_norm_kernel<8>, 8);
}

}  // namespace shai
