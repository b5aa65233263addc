// Fold of split-K partial sums, residual and the next row norm in one launch.
//
// A layer of a small batch is a chain of launches that cost 3.5 to 4.5 us each whatever they do: a product whose K is split over
// workgroups, its fold, the norm of the result, the next product.  The fold and the norm read some hundred KB; here a wave takes
// a row, all its loads issued before the first addition, and the row never leaves its registers between the two.
// 154 x 1024 x 4096: product, fold and norm 13.9 us -> 10.9, 197 x 768 x 3072 13.5 -> 10.2, 32 x 768 x 3072 11.6 -> 8.6, 512 x 1280 x 5120 25.2 ->
// 21.3; where K was not split before, splitting it pays now: 197 x 768 x 768 8.6 -> 7.9, 32 x 768 x 768 10.0 -> 6.9.
#include "fold_norm.h"
#include "common.h"
#include "launch.h"

namespace shai {

namespace {

__device__ __forceinline__ float at4(const uint2_& t, int e) { return bf2f(e & 1 ? t[e >> 1] >> 16 : t[e >> 1] & 0xffff); }

__device__ __forceinline__ uint2_ pack4(const float (&f)[4]) { return uint2_{pack2(f[0], f[1]), pack2(f[2], f[3])}; }

// NC: 256-column chunks of a row, 4 columns a lane each.  The parts are added in the order, and the bias and the residual with the
// operations, of gemm_splitk_reduce: y has the bits that it writes.
template <int NC>
__global__ void __launch_bounds__(64) fold_norm_kernel(const FoldNormArgs p) {
  constexpr int ROUND = NC <= 4 ? 4 : 2;   // parts in flight
  const int lane = threadIdx.x;
  const long row = blockIdx.x, slab = (long)p.rows * p.D;
  const float* src = p.parts + row * p.D;
  float v[NC][4];
  uint2_ r[NC], bias[NC], gain[NC], shift[NC];
  bool in[NC];
  int col[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    in[c] = (c * 64 + lane) * 4 < p.D;
    col[c] = in[c] ? (c * 64 + lane) * 4 : 0;   // spare lanes read column 0
#pragma unroll
    for (int e = 0; e < 4; ++e) v[c][e] = 0.f;
    auto load = [&](const bf16_t* at) { return *reinterpret_cast<const uint2_*>(at + col[c]); };
    const uint2_ one = {0x3f803f80u, 0x3f803f80u}, zero = {0u, 0u};
    r[c] = p.residual ? load(p.residual + row * p.ldr) : zero;
    bias[c] = p.bias ? load(p.bias) : zero;
    gain[c] = p.gamma ? load(p.gamma) : one;
    shift[c] = p.beta ? load(p.beta) : zero;
  }
  for (int s0 = 0; s0 < p.splits; s0 += ROUND) {
    float4_ x[ROUND][NC];
#pragma unroll
    for (int u = 0; u < ROUND; ++u)
#pragma unroll
      for (int c = 0; c < NC; ++c)
        x[u][c] = s0 + u < p.splits ? *reinterpret_cast<const float4_*>(src + (s0 + u) * slab + col[c]) : float4_{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < ROUND; ++u)
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[c][e] += x[u][c][e];
  }
  float sum = 0.f, sq = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (p.bias) v[c][e] += at4(bias[c], e);
      if (p.residual) v[c][e] += at4(r[c], e) * p.res_alpha;
    }
    const uint2_ w = pack4(v[c]);
    if (in[c]) *reinterpret_cast<uint2_*>(p.y + row * p.D + col[c]) = w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[c][e] = in[c] ? at4(w, e) : 0.f;   // as the next layer reads it
      sum += v[c][e];
      sq += v[c][e] * v[c][e];
    }
  }
  float mean = 0.f, rstd;
  if (p.rms) {
    rstd = rsqrtf(wave_sum(sq) / p.D + p.eps);
  } else {
    mean = wave_sum(sum) / p.D;
    float var = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float d = in[c] ? v[c][e] - mean : 0.f;
        var += d * d;
      }
    rstd = rsqrtf(wave_sum(var) / p.D + p.eps);
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[c][e] = (v[c][e] - mean) * rstd * at4(gain[c], e) + at4(shift[c], e);
    if (in[c]) *reinterpret_cast<uint2_*>(p.out + row * p.D + col[c]) = pack4(v[c]);
  }
}

}  // namespace

bool fold_norm_supported(const FoldNormArgs& a) {
  const uintptr_t at = (uintptr_t)a.bias | (uintptr_t)a.residual | (uintptr_t)a.y | (uintptr_t)a.gamma | (uintptr_t)a.beta | (uintptr_t)a.out;
  return a.D % 4 == 0 && a.D <= 2048 && (at & 7) == 0 && (a.residual == nullptr || a.ldr % 4 == 0);
}

hipError_t launch_fold_norm(const FoldNormArgs& a, hipStream_t s) {
  if (a.rows == 0) return hipSuccess;
  if (!fold_norm_supported(a)) return hipErrorInvalidValue;
  const int chunks = (a.D + 255) / 256;
  return launch(chunks <= 1   ? fold_norm_kernel<1>
                : chunks <= 2 ? fold_norm_kernel<2>
                : chunks <= 3 ? fold_norm_kernel<3>
                : chunks <= 4 ? fold_norm_kernel<4>
                : chunks <= 5 ? fold_norm_kernel<5>
                              : fold_norm_kernel<8>,
                a.rows, 64, s, a);
}

}  // namespace shai
