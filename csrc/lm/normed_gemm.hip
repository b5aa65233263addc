// C = epi(norm(x + sum of a sublayer's parts) W^T) of a decode step's few rows, and x + parts for the next layer.
//
// The norm of one row is 2.7 us on one CU, 4.7 with its launch, and the product behind it waits for all of it.  Here every workgroup makes
// the norm itself: the row, its parts and the gain are asked for first (8 (2 + parts) KB of a row of 2048, from the XCD's L2), the first weights
// right behind them, and these travel while the norm is made.  The first workgroup writes the residual (to memory that no workgroup reads).
//
// A workgroup takes every gridDim-th tile of 16 rows of W, so that the norm is made once for all of them (one tile a workgroup: 1089 norms,
// 19.1 us for 1 x 17424 x 2048 where norm and product apart take 19.4; 256 workgroups 20.8, 512 17.7, 1024 18.6).  Eight waves split
// K in steps of 64, and a wave's steps follow each other across tiles through a ring of D in registers: the end of a tile, where the
// waves' sums meet in LDS, has the next one's weights beside it.
#include "lm_device.h"
#include "normed_gemm.h"

namespace shai_lm {

namespace {

constexpr int NW = 8, NT = 512;           // waves, threads
constexpr int kGrid = 512;                // two workgroups for each CU: every form that is compiled has at most 128 registers

template <typename O, int M, int NV, bool MANY>   // NV: groups of 4 columns a thread and row has; MANY: more than four parts
__global__ void __launch_bounds__(NT, 2) normed_gemm_kernel(const NormedGemmArgs p) {
  constexpr int D = 8;
  __shared__ __attribute__((aligned(16))) bf16_t h[M][NV * NT * 4];
  __shared__ float4_ red[2][NW][64];
  __shared__ float sums[NW][M];
  const GemmArgs& g = p.g;
  const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int K = g.K, per = (K / 64 + NW - 1) / NW;              // steps of a wave and tile; the last may lie past K
  const int all = (g.N + 15) / 16, tiles = (all - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const bf16_t* W = static_cast<const bf16_t*>(g.W);
  uint4_ w[D][2];
  int f_tile = blockIdx.x, f_at = 0;                            // where the ring's next fetch lies
  auto fetch = [&](int u) {
    if (f_tile < all) {
      const int k = min(f_at * NW + wid, K / 64 - 1) * 64;      // (multiplied by zeros past K)
      const bf16_t* at = W + (long)min(f_tile * 16 + r, g.N - 1) * K + k + q * 16;
      w[u][0] = *reinterpret_cast<const uint4_*>(at);
      w[u][1] = *reinterpret_cast<const uint4_*>(at + 8);
    }
    if (++f_at == per) f_at = 0, f_tile += gridDim.x;
  };
  // What the norm needs is asked for first: loads return in order, and behind the ring's it would wait for those to come from memory.
  float4_ v[M][NV], gain[NV], d[M][NV][MANY ? 8 : 4];
  constexpr int P = MANY ? 8 : 4;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = min((i * NT + tid) * 4, K - 4);               // spare threads read the last columns
    gain[i] = load4(p.w + c);
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const long at = (long)min(m, g.M - 1) * K + c;
      if (p.x) v[m][i] = load4(p.x + at);
      else v[m][i] = load4(static_cast<const bf16_t*>(p.table) + (long)min(max(p.ids[min(m, g.M - 1)], 0), p.V - 1) * K + c) * p.scale;
      if (p.delta) {
#pragma unroll
        for (int j = 0; j < P; ++j) d[m][i][j] = load4(p.delta + min(j, p.parts - 1) * p.part_stride + at);
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < D; ++u) fetch(u);
  __builtin_amdgcn_sched_barrier(0);
  // the parts are added in residual_norm's order
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * NT + tid) * 4;
    const float4_ zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < M; ++m) {
      if (p.delta) {
        float4_ t = d[m][i][0];
        if constexpr (MANY) {
#pragma unroll
          for (int j = 1; j < P; ++j) t += j < p.parts ? d[m][i][j] : zero;
        } else {
          t += (1 < p.parts ? d[m][i][1] : zero) + (2 < p.parts ? d[m][i][2] : zero) + (3 < p.parts ? d[m][i][3] : zero);
        }
        v[m][i] += t;
      }
      if (c >= K || m >= g.M) v[m][i] = zero;
      else if (p.x_out && blockIdx.x == 0) store4(p.x_out + (long)m * K + c, v[m][i]);
    }
  }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) ss += v[m][i][0] * v[m][i][0] + v[m][i][1] * v[m][i][1] + v[m][i][2] * v[m][i][2] + v[m][i][3] * v[m][i][3];
    ss = wave_sum(ss);
    if (lane == 0) sums[wid][m] = ss;
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < M; ++m) {
    float ss = 0.f;
#pragma unroll
    for (int u = 0; u < NW; ++u) ss += sums[u][m];
    const float f = 1.f / sqrtf(ss * (1.f / (float)p.width) + p.eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) store4(&h[m][(i * NT + tid) * 4], v[m][i] * f * gain[i]);
  }
  __syncthreads();

  const bf16_t* row = &h[min(r, M - 1)][q * 16];
  float4_ acc = {0.f, 0.f, 0.f, 0.f};
  int tile = 0, at = 0;
  auto use = [&](int u) {
    const int s = at * NW + wid;
    if (s < K / 64) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[u][j]),
                                                      *reinterpret_cast<const bf16x8*>(row + s * 64 + 8 * j), acc, 0, 0, 0);
    }
    if (++at < per) return;
    const int buf = tile & 1;                                   // the buffer before is read by now: a barrier lies between
    red[buf][wid][lane] = acc;
    acc = float4_{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    if (wid == (tile & (NW - 1))) {
      float4_ c = red[buf][0][lane];
#pragma unroll
      for (int i = 1; i < NW; ++i) c += red[buf][i][lane];
      if (r < g.M) store_cols<O, EC_PLAIN>(g, static_cast<O*>(g.C), r, ((int)blockIdx.x + tile * (int)gridDim.x) * 16 + 4 * q, c);
    }
    at = 0;
    ++tile;
  };
  const int total = tiles * per;
  for (int i = 0; i < total; i += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      if (i + u < total) {
        use(u);
        fetch(u);
      }
    }
  }
}

template <typename O>
void rows(const NormedGemmArgs& a, hipStream_t s) {
  const int tiles = (a.g.N + 15) / 16, grid = tiles < kGrid ? tiles : kGrid;
  auto go = [&](auto kernel) { kernel<<<grid, NT, 0, s>>>(a); };
  if (a.g.M == 2) go(normed_gemm_kernel<O, 2, 1, false>);
  else if (a.g.K > NT * 4) go(normed_gemm_kernel<O, 1, 2, false>);
  else if (a.parts > 4) go(normed_gemm_kernel<O, 1, 1, true>);
  else go(normed_gemm_kernel<O, 1, 1, false>);
}

}  // namespace

// The forms of which a CU holds two workgroups.  us apart and in one launch, bf16 outputs of 17424 columns: one row of 2048 in four parts 19.3 and
// 17.7, in eight 19.6 and 18.7, of 4096 in four 31.7 and 29.8; two rows of 2048 in four 19.5 and 19.1.  The others need 147 to 224 registers: one
// row of 4096 in eight parts 32.2 and 36.7, two of 2048 in eight 19.8 and 22.7, two of 4096 32.2 and 37.3; four rows of 2048 20.6 and 22.8.
bool normed_gemm_fits(int M, int K, int parts) {
  return K % 64 == 0 && (M == 1 ? parts <= 4 ? K <= 4096 : parts <= 8 && K <= 2048 : M == 2 && parts <= 4 && K <= 2048);
}

void launch_normed_gemm(const NormedGemmArgs& a, hipStream_t s) {
  if (a.g.out_f32) rows<float>(a, s);
  else rows<bf16_t>(a, s);
  SHAI_CHECK_LAUNCH();
}

}  // namespace shai_lm
