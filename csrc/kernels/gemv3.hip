// Skinny GEMM without a split over workgroups ("skinny3", M <= 16 activation rows):
//
//   C[m, n] = act(alpha * sum_k X[m, k] * W[n, k] + bias[n]) (+ res_alpha * R[m, n])
//
// gemv.hip and gemv2.hip have tiles of 64 and 128 weight rows: a matrix of a few thousand rows fills the chip only with K cut over
// workgroups, and the partial sums then cost a fold, in a launch of its own or by the last workgroup of a tile.  Here a workgroup has 16
// weight rows and all of K, so 4096 rows are one workgroup for each of the 256 CUs, and the sums never leave it.
//
// * Eight waves cut K among them in units of 64, one 128-byte line of each weight row: unit u belongs to wave u % 8.  Weights and
//   activations go straight to registers (v_mfma_f32_16x16x32_bf16: 16 weight rows as A, the activation rows as B, 16 bytes a lane and
//   operand).  The waves share nothing before the end, so there is no barrier in the loop, and a ring of 8 steps keeps 8 KB of W a wave
//   in flight.
// * Every workgroup reads all activations, from its XCD's L2: M / 16 bytes for a byte of W.  That is why it ends at 16 rows: at 32 the
//   activations are twice the weights and bound it (4096 x 4096 16.0 us, gemv.hip 11.5; 1024 x 2816 12.1 and 7.9).  Rows past M or N and
//   columns past K are zeros of the buffer descriptor and cost no traffic.
// * The waves' sums meet in LDS and are added in wave order.
//
// Bound by the weights' way from memory where there are enough of them, by latency below.  us a product with its fold, cold weights, the
// best of gemv.hip's forms and this, one row: 768 x 768 5.6 -> 4.2, 1024 x 1024 5.7 -> 4.4, 4096 x 4096 10.5 -> 9.4 (3.6 TB/s), 3072 x 1024
// 7.0 -> 4.9; a K of several times the rows is better cut over workgroups (4096 x 14336 22.9 and 25.8).
#include "common.h"
#include "launchers.h"

namespace shai {

namespace {

typedef __bf16 bf16x8t __attribute__((ext_vector_type(8)));

constexpr int S3_BN = 16;                  // weight rows of a workgroup, and most activation rows
constexpr int S3_WAVES = 8;
constexpr int S3_DEPTH = 8;                // steps of 32 in flight, two to a unit
constexpr uint32_t S3_OOB = 0x80000000u;   // past the end of any operand, with the step's bytes added too: reads zeros

__device__ __forceinline__ __amdgpu_buffer_rsrc_t s3_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

__global__ void __launch_bounds__(S3_WAVES * 64) skinny3_kernel(const GemmArgs p) {
  __shared__ __attribute__((aligned(16))) float red[S3_WAVES][16][S3_BN + 4];
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = blockIdx.x * S3_BN;
  const int units = (p.K + 63) >> 6;
  const int steps = 2 * ((units + S3_WAVES - 1) / S3_WAVES);
  const __amdgpu_buffer_rsrc_t rW = s3_rsrc(p.W, (uint32_t)((long)p.N * p.ldw * 2));
  const __amdgpu_buffer_rsrc_t rX = s3_rsrc(p.A, (uint32_t)((long)p.M * p.lda * 2));
  const uint32_t wbase = n0 + r < p.N ? (uint32_t)(((long)(n0 + r) * p.ldw + q * 8) * 2) : S3_OOB;
  const uint32_t xbase = r < p.M ? (uint32_t)(((long)r * p.lda + q * 8) * 2) : S3_OOB;

  uint4_ wf[S3_DEPTH], xf[S3_DEPTH];
  auto load = [&](int slot, int step) {
    const int k = ((step >> 1) * S3_WAVES + w) * 64 + (step & 1) * 32;
    const bool in = k + q * 8 < p.K;
    wf[slot] = __builtin_bit_cast(uint4_, __builtin_amdgcn_raw_buffer_load_b128(rW, in ? wbase + 2u * k : S3_OOB, 0, 2));   // read once: nt
    xf[slot] = __builtin_bit_cast(uint4_, __builtin_amdgcn_raw_buffer_load_b128(rX, in ? xbase + 2u * k : S3_OOB, 0, 0));
  };
  float4_ acc = {0.f, 0.f, 0.f, 0.f};
  auto use = [&](int slot) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8t, wf[slot]), __builtin_bit_cast(bf16x8t, xf[slot]), acc, 0, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < S3_DEPTH; ++i) load(i, i);   // steps past the end read zeros
  for (int base = 0; base + S3_DEPTH < steps; base += S3_DEPTH) {
#pragma unroll
    for (int i = 0; i < S3_DEPTH; ++i) {
      use(i);
      load(i, base + S3_DEPTH + i);
    }
  }
#pragma unroll
  for (int i = 0; i < S3_DEPTH; ++i) use(i);

  *reinterpret_cast<float4_*>(&red[w][r][4 * q]) = acc;   // columns 4 q .. 4 q + 3 of activation row r
  __syncthreads();
  if (tid >= 64) return;
  const int m = tid >> 2, n = n0 + 4 * (tid & 3);
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < S3_WAVES; ++u) {
    const float4_ a = *reinterpret_cast<const float4_*>(&red[u][m][4 * (tid & 3)]);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += a[e];
  }
  if (m >= p.M || n >= p.N) return;
  bf16_t* c = p.C + (long)m * p.ldc + n;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = apply_act_rt(p.act, v[e] * p.alpha + (p.bias ? bf2f(p.bias[n + e]) : 0.f));
    if (p.residual) v[e] += bf2f(p.residual[(long)m * p.ldr + n + e]) * p.res_alpha;
  }
  if (((uintptr_t)c & 7) == 0) {
    *reinterpret_cast<uint2_*>(c) = uint2_{pack2(v[0], v[1]), pack2(v[2], v[3])};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) c[e] = f2bf(v[e]);
  }
}

}  // namespace

bool skinny3_supported(const GemmArgs& a) {
  return a.M >= 1 && a.M <= 16 && !a.conv && !a.glu && !a.rms && a.batch <= 1 && a.w_slice_rows == 0 && a.w_scale == nullptr &&
         a.bias2d == nullptr && a.gate == nullptr && a.in_scale == nullptr && a.row_mr == nullptr && a.K % 8 == 0 && a.N % 4 == 0 &&
         a.lda % 8 == 0 && a.ldw % 8 == 0 && (long)a.N * a.ldw * 2 < 0x7fffffffL && (long)a.M * a.lda * 2 < 0x7fffffffL;
}

void launch_skinny3(const GemmArgs& a, hipStream_t s) {
  skinny3_kernel<<<(a.N + S3_BN - 1) / S3_BN, S3_WAVES * 64, 0, s>>>(a);
}

}  // namespace shai
