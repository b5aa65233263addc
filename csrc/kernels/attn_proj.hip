// Attention of short sequences (up to 256 keys, heads of 64) and the output projection of every head, in one launch.
//
// In a layer of a small batch each launch costs 4 to 8 us whatever it does, and attention, projection, fold and norm were four.  The
// projection's K is the heads: a workgroup that has a head's output of 64 rows multiplies it by that head's 64 columns of W, and the
// sums over heads are left to the launch that makes the next norm (fold_norm.hip), which adds partial sums anyway.
//
// * Workgroup: 64 queries of a head (16 a wave) and 256 columns of W.  The attention is made again for every 256 columns: it is a few
//   dozen MFMAs a wave, and the columns would otherwise be one workgroup's to read.
// * All loads (q, k, v, W, bias) are issued before anything is waited for: K and V lie whole in LDS, W's 4 tiles a wave in registers.
// * Scores come as S^T = K Q^T (v_mfma_f32_16x16x32_bf16), so a lane has one query's scores; P feeds O^T = V^T P^T from the registers
//   it is made in (keys in the order in which the lanes hold them), V^T by transposed LDS reads.  O passes LDS as bf16, the rounding of
//   attention's output in memory, and every wave multiplies all 64 rows by its columns.
//
// us with cold weights, attention, product and fold with norm -> here with the fold: 16 heads to 1024 columns, 7 rows 12.2 -> 8.2, 32 rows
// 11.3 -> 8.9, 77 rows 14.3 -> 11.8, 128 rows 15.9 -> 14.5, 2 x 77 rows 14.9 -> 14.1; 12 heads to 768, 197 rows 15.9 -> 15.5.  From there the
// partial sums, a row's outputs of every head in fp32, cost more than the launch (200 rows 15.6 -> 16.4, 256 rows 14.4 -> 17.7); two heads to
// a workgroup halve them but follow each other (32 rows 10.4, 128 rows 15.2, 256 rows 15.7).
#include "attn_proj.h"
#include "common.h"
#include "launch.h"

namespace shai {

namespace {

typedef __bf16 bf16x8p __attribute__((ext_vector_type(8)));
typedef short s4p __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4p lds_s4p;

constexpr int kRow = 72;       // elements of a row of 64 in LDS: rows 36 banks apart, no conflicts on fragments of 16 rows
constexpr int kCols = 256;     // columns of W a workgroup has
constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float4_ mma(const uint4_& a, const uint4_& b, float4_ c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8p, a), __builtin_bit_cast(bf16x8p, b), c, 0, 0, 0);
}

// NK: key tiles of 64.  BIAS: 0 none, 1 any, 2 rows of 4 aligned values.
template <int NK, int BIAS>
__global__ void __launch_bounds__(256) attn_proj_kernel(const AttnProjArgs p) {
  constexpr int T = 4 * NK;    // tiles of 16 keys
  __shared__ __attribute__((aligned(16))) bf16_t sk[NK * 64 * kRow], sv[NK * 64 * kRow], so[64 * kRow];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r = lane & 15, g = lane >> 4;
  const int blocks = (p.Sq + 63) / 64, b = blockIdx.x / blocks, q0 = (blockIdx.x - b * blocks) * 64;
  const int h = blockIdx.y, n0 = blockIdx.z * kCols + w * 64;
  const int qi = q0 + 16 * w + r;                              // this lane's query
  const int kv_len = p.kv_lens ? min(p.kv_lens[b], p.Skv) : p.Skv;
  const int row = tid >> 3, c8 = (tid & 7) * 8;                // of the keys and values that this thread stages
  const uint4_ zero = {0u, 0u, 0u, 0u};

  uint4_ kk[2 * NK], vv[2 * NK], q[2], wf[4][2];
  {
    const bf16_t* k = p.k + (long)b * p.k_bs + h * 64 + c8;
    const bf16_t* v = p.v + (long)b * p.v_bs + h * 64 + c8;
#pragma unroll
    for (int i = 0; i < 2 * NK; ++i) {                         // rows past the end are read at the last one and stored as zeros
      const int at = min(row + 32 * i, p.Skv - 1);
      kk[i] = *reinterpret_cast<const uint4_*>(k + at * p.k_ts);
      vv[i] = *reinterpret_cast<const uint4_*>(v + at * p.v_ts);
    }
    const bf16_t* qp = p.q + (long)b * p.q_bs + (long)min(qi, p.Sq - 1) * p.q_ts + h * 64 + 8 * g;
#pragma unroll
    for (int u = 0; u < 2; ++u) q[u] = *reinterpret_cast<const uint4_*>(qp + 32 * u);
  }
  [[maybe_unused]] uint2_ bias[BIAS ? T : 1];
  if constexpr (BIAS != 0) {
    const bf16_t* at = p.bias + ((long)h * p.Sq + min(qi, p.Sq - 1)) * p.Skv;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int key = 16 * t + 4 * g;
      if constexpr (BIAS == 2) {
        bias[t] = *reinterpret_cast<const uint2_*>(at + min(key, p.Skv - 4));
      } else {
        uint32_t e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = at[min(key + i, p.Skv - 1)];
        bias[t] = uint2_{e[0] | e[1] << 16, e[2] | e[3] << 16};
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
      wf[t][u] = *reinterpret_cast<const uint4_*>(p.W + (long)min(n0 + 16 * t + r, p.N - 1) * p.ldw + h * 64 + 32 * u + 8 * g);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < 2 * NK; ++i) {
    const int at = row + 32 * i;
    *reinterpret_cast<uint4_*>(&sk[at * kRow + c8]) = at < kv_len ? kk[i] : zero;
    *reinterpret_cast<uint4_*>(&sv[at * kRow + c8]) = at < kv_len ? vv[i] : zero;
  }
  __syncthreads();

  // scores of query r: s[t][i] of key 16 t + 4 g + i, to the base 2
  float4_ s[T];
  float m = -INFINITY;
#pragma unroll
  for (int t = 0; t < T; ++t) {
    s[t] = float4_{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 2; ++u) s[t] = mma(*reinterpret_cast<const uint4_*>(&sk[(16 * t + r) * kRow + 32 * u + 8 * g]), q[u], s[t]);
  }
#pragma unroll
  for (int t = 0; t < T; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = 16 * t + 4 * g + i;
      float x = s[t][i] * p.scale;
      if constexpr (BIAS != 0) x += bf2f(i & 1 ? bias[t][i >> 1] >> 16 : bias[t][i >> 1] & 0xffff);
      s[t][i] = key < kv_len && (!p.causal || key <= qi) ? x * kLog2e : -INFINITY;
      m = fmaxf(m, s[t][i]);
    }
  m = fmaxf(m, __shfl_xor(m, 16, 64));
  m = fmaxf(m, __shfl_xor(m, 32, 64));
  if (m == -INFINITY) m = 0.f;                                 // no key at all: an output of zeros
  float l = 0.f;
  uint4_ pf[T / 2];
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[t][i] = __builtin_amdgcn_exp2f(s[t][i] - m);
      l += s[t][i];
    }
    pf[t >> 1][2 * (t & 1)] = pack2(s[t][0], s[t][1]);
    pf[t >> 1][2 * (t & 1) + 1] = pack2(s[t][2], s[t][3]);
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  // O^T, 16 columns of V at a time.  A step of 32 keys takes them as P has them: lane group g its keys 4 g .. 4 g + 3 of both tiles.
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int tq = r >> 2, tp = r & 3;                           // a transposed read gives 16 lanes 4 rows x 16 columns
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    float4_ o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < T / 2; ++u) {
      bf16_t* at = &sv[(32 * u + 4 * g + tq) * kRow + 16 * d + 4 * tp];
      const s4p lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4p*)at);
      const s4p hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4p*)(at + 16 * kRow));
      const uint2_ a = __builtin_bit_cast(uint2_, lo), c = __builtin_bit_cast(uint2_, hi);
      o = mma(uint4_{a[0], a[1], c[0], c[1]}, pf[u], o);
    }
    *reinterpret_cast<uint2_*>(&so[(16 * w + r) * kRow + 16 * d + 4 * g]) = uint2_{pack2(o[0] * inv, o[1] * inv), pack2(o[2] * inv, o[3] * inv)};
  }
  __syncthreads();

  const long rows = (long)p.B * p.Sq;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int at = q0 + 16 * j + r;
    const uint4_ x0 = *reinterpret_cast<const uint4_*>(&so[(16 * j + r) * kRow + 8 * g]);
    const uint4_ x1 = *reinterpret_cast<const uint4_*>(&so[(16 * j + r) * kRow + 32 + 8 * g]);
    float* out = p.parts + (h * rows + (long)b * p.Sq + at) * p.N;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int n = n0 + 16 * t + 4 * g;
      const float4_ y = mma(wf[t][1], x1, mma(wf[t][0], x0, float4_{0.f, 0.f, 0.f, 0.f}));
      if (at < p.Sq && n < p.N) *reinterpret_cast<float4_*>(out + n) = y;
    }
  }
}

template <int NK>
hipError_t go(const AttnProjArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * ((a.Sq + 63) / 64)), a.H, (a.N + kCols - 1) / kCols);
  auto* kernel = a.bias == nullptr ? attn_proj_kernel<NK, 0>
                 : a.Skv % 4 == 0 && ((uintptr_t)a.bias & 7) == 0 ? attn_proj_kernel<NK, 2> : attn_proj_kernel<NK, 1>;
  AttnProjArgs p = a;
  void* args[] = {&p};
  return hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, dim3(256), args, 0, s);
}

}  // namespace

bool attn_proj_supported(const AttnProjArgs& a) {
  const uintptr_t at = (uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.W | (uintptr_t)a.parts;
  const long strides = a.q_bs | a.q_ts | a.k_bs | a.k_ts | a.v_bs | a.v_ts | a.ldw;
  return a.B >= 1 && a.H >= 1 && a.H <= 65535 && a.Sq >= 1 && a.Skv >= 1 && a.Skv <= 256 && a.N >= 16 && a.N % 16 == 0 && a.N <= 65535 * kCols &&
         (long)a.B * a.Sq <= 1 << 24 && (at & 15) == 0 && (strides & 7) == 0;
}

hipError_t launch_attn_proj(const AttnProjArgs& a, hipStream_t s) {
  if (!attn_proj_supported(a)) return hipErrorInvalidValue;
  return a.Skv <= 64 ? go<1>(a, s) : a.Skv <= 128 ? go<2>(a, s) : go<4>(a, s);
}

}  // namespace shai
