// C = A W^T in bf16 for tiles that fill the chip (prefill): 256 x 256 tiles of four waves, each 128 x 128, one wave per SIMD.
//
// What bounds the eight-wave tile of gemm_tile.hip: per 64-wide k-tile its waves (128 x 64 each) read 192 KB of fragments out of
// LDS, and all of them drain their loads and meet before the next one.  A 128 x 128 wave tile reads 128 KB, and the wave hides its
// own latencies: fragments live in two register sets, one k-step being multiplied while the other is read.  Per k-tile t
//   (a) MFMAs of k-step 0 beside the reads of k-step 1;
//   (b) this wave's DMA of tile t + 1 has landed, its reads of tile t are done; one barrier makes both true of every wave;
//   (c) MFMAs of k-step 1 beside the DMA of tile t + 2 into the stage just left and the reads of tile t + 1's k-step 0.
// Tiles left over after whole rounds of the 256 CUs, up to half a round, are cut in quarters (128 x 128, four k-tiles in flight):
// a quarter takes about 0.35 of a round, so one or two of them per CU are shorter than a round that leaves most of the chip idle.
// Measured, M x N x K, us (eight-wave tile -> this without quarters -> with): 8192 x 8192 x 8192 914 -> 821 (1339 TF/s),
// 7700 x 2048 x 4096 122 -> 117; 7700 x 14848 x 2048 (22 tiles left) 451 -> 433 -> 411, 8192 x 16640 x 2048 (32) 543 -> 511 -> 481,
// 4096 x 4608 x 2048 (32) 103 -> 102 -> 73, 4096 x 6144 x 2048 (128) 109 -> 104 -> 97.
#include "lm_device.h"
#include "lm.h"

#include <type_traits>
#include <utility>

namespace shai_lm {

namespace {

constexpr uint32_t kOob = 0x80000000u;           // beyond any buffer: reads as zero, also with a k offset added
constexpr int kTile = 256, kLds = 128 * (kTile + 4) * 4;   // LDS: the fp32 rows of the epilogue; the k-tiles take 128 KB of it

// the order the scheduler is to keep per group of NB MFMAs: DMA, fragment reads in the first half of the groups, MFMAs
template <int NB, int DMA, int... G>
__device__ __forceinline__ void interleave(std::integer_sequence<int, G...>) {
  const auto group = [](auto g) {
    if constexpr (DMA > 0) __builtin_amdgcn_sched_group_barrier(0x020, DMA, 0);
    if constexpr (decltype(g)::value < NB / 2) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
    __builtin_amdgcn_sched_group_barrier(0x008, NB, 0);
  };
  (group(std::integral_constant<int, G>{}), ...);
}

// One tile of 32 NB x 32 NB at (m0, n0), waves of 16 NB x 16 NB; ST k-tiles in LDS.
template <int NB, int ST>
__device__ __forceinline__ void tile(const GemmArgs& p, bf16_t* smem, int m0, int m_end, int n0, const bf16_t* Wt) {
  constexpr int B = 32 * NB, FR = 2 * NB, STAGE = 2 * B * 64, LD = B + 4;
  static_assert(ST * STAGE * 2 <= kLds && 16 * NB * LD * 4 <= kLds && (ST & (ST - 1)) == 0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const __amdgpu_buffer_rsrc_t rW = rsrc(Wt, (long)p.N * p.K * 2), rA = rsrc(p.A, ((long)(p.a_rows - 1) * p.lda + p.K) * 2);

  // byte offset of this lane's 16-byte chunk of the NB + NB row groups its wave stages, at k = 0; the bank swizzle is on the source
  const int lrow = lane >> 3, lpos = lane & 7;
  uint32_t off[FR];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int r = wid * (B / 4) + j * 8 + lrow, ch = (lpos ^ ((r >> 1) & 7)) * 8, m = m0 + r, n = n0 + r;
    const long src = m < m_end ? (p.gather ? p.gather[m] : m) : -1;
    off[j] = src < 0 ? kOob : (uint32_t)((src * p.lda + ch) * 2);
    off[NB + j] = n < p.N ? (uint32_t)(((long)n * p.K + ch) * 2) : kOob;
  }
  const int nk = p.K / 64;
  // row group g of k-tile t (all zeros past the last tile: every tile's loads are counted alike)
  auto dma = [&](int t, int g) {
    bf16_t* dst = smem + (t & (ST - 1)) * STAGE + ((g < NB ? 0 : B) + wid * (B / 4) + (g % NB) * 8) * 64;
    dma16(g < NB ? rA : rW, dst, (off[g] + (uint32_t)t * 128u) | (t < nk ? 0u : kOob));
  };
  // fragment f of k-step s: W's blocks of 16 rows first, the first MFMAs need all of them
  const int fr = lane & 15, fq = lane >> 4;
  typedef bf16x8 Set[FR];
  auto read = [&](int t, int s, int f, Set& x) {
    const int row = f < NB ? B + wn * (B / 2) + 16 * f : wm * (B / 2) + 16 * (f - NB);
    x[f] = *reinterpret_cast<const bf16x8*>(smem + (t & (ST - 1)) * STAGE + (row + fr) * 64 + (((fq + 4 * s) ^ ((fr >> 1) & 7)) << 3));
  };
  // a set is redefined after its inline wait: the compiler's own wait counts do not see that one
  auto landed = [](Set& x) {
#pragma unroll
    for (int f = 0; f < FR; ++f) asm volatile("" : "+v"(x[f]));
  };

  float4_ acc[NB][NB];
  Set x0, x1;
#pragma unroll
  for (int g = 0; g < ST * FR; ++g) dma(g / FR, g % FR);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 1) * FR) : "memory");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int f = 0; f < FR; ++f) read(0, 0, f, x0);

  auto half0 = [&](int t, auto first) {
#pragma unroll
    for (int g = 0; g < NB; ++g) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (g < NB / 2) read(t, 1, 4 * g + u, x1);
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[g][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x0[j], x0[NB + g], decltype(first)::value ? float4_{} : acc[g][j], 0, 0, 0);
    }
    interleave<NB, 0>(std::make_integer_sequence<int, NB>{});
    __builtin_amdgcn_sched_barrier(0);
  };
  auto half1 = [&](int t) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((ST - 2) * FR) : "memory");
    landed(x1);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NB; ++g) {
      dma(t + ST, 2 * g);
      dma(t + ST, 2 * g + 1);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (g < NB / 2) read(t + 1, 0, 4 * g + u, x0);
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[g][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x1[j], x1[NB + g], acc[g][j], 0, 0, 0);
    }
    interleave<NB, 2>(std::make_integer_sequence<int, NB>{});
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    landed(x0);
  };
  half0(0, std::true_type{});
  for (int t = 0; t + 1 < nk; ++t) {
    half1(t);
    half0(t + 1, std::false_type{});
  }
  half1(nk - 1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // The tile goes through LDS as fp32, one wave row at a time, so that a wave stores whole lines: 16 bytes a lane where
  // rows allow it and no side columns are among them.  (A store per block of the accumulators would unroll the epilogue 64 times.)
  bf16_t* C = static_cast<bf16_t*>(p.C);
  float* buf = reinterpret_cast<float*>(smem);
  const bool lines = p.ldc % 8 == 0 && p.n_main % 8 == 0 && (p.n_main == p.N || n0 + B <= p.n_main);
  for (int h = 0; h < 2; ++h) {
    __syncthreads();
    if (wm == h) {
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) store4(buf + (16 * i + fr) * LD + wn * (B / 2) + 16 * j + 4 * fq, acc[i][j]);
    }
    __syncthreads();
    const int mh = m0 + B / 2 * h;
    if (lines) {
      for (int id = tid; id < B / 2 * (B / 8); id += 256) {
        const int r = id / (B / 8), n = id % (B / 8) * 8, m = mh + r;
        if (m >= m_end || n0 + n >= p.n_main) continue;
        float4_ u = load4(buf + r * LD + n), v = load4(buf + r * LD + n + 4);
        epilogue_cols<bf16_t, EC_PLAIN>(p, m, n0 + n, u);
        epilogue_cols<bf16_t, EC_PLAIN>(p, m, n0 + n + 4, v);
        *reinterpret_cast<uint4_*>(C + (long)m * p.ldc + n0 + n) =
            uint4_{pack2(u[0], u[1]), pack2(u[2], u[3]), pack2(v[0], v[1]), pack2(v[2], v[3])};
      }
    } else {
      for (int id = tid; id < B / 2 * (B / 4); id += 256) {
        const int r = id / (B / 4), n = id % (B / 4) * 4;
        if (mh + r < m_end) store_cols<bf16_t, EC_PLAIN>(p, C, mh + r, n0 + n, load4(buf + r * LD + n));
      }
    }
  }
}

}  // namespace

// Workgroups 0 .. whole - 1 take one tile each, every four behind them the quarters of one of the remaining tiles.
__global__ void __launch_bounds__(256, 1) gemm_wide_kernel(const GemmArgs p, int whole) {
  extern __shared__ __attribute__((aligned(16))) bf16_t smem[];
  const int tiles_m = p.tiles ? p.n_tiles : (p.M + kTile - 1) / kTile, tiles_n = (p.N + kTile - 1) / kTile;
  int bid = blockIdx.x, part = 0;
  const bool quarter = bid >= whole;
  if (quarter) {
    part = (bid - whole) & 3;
    bid = whole + ((bid - whole) >> 2);
  } else {
    const int xcd = bid & 7, q = whole >> 3, r = whole & 7;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (bid >> 3);
  }
  constexpr int GROUP = 8;
  const int group = bid / (GROUP * tiles_n), first_m = group * GROUP;
  const int gsize = min(tiles_m - first_m, GROUP);
  const int in_group = bid - group * GROUP * tiles_n;
  const int mt = first_m + in_group % gsize, n0 = (in_group / gsize) * kTile;
  if (quarter) {
    const int m = mt * kTile + (part >> 1) * 128, n = n0 + (part & 1) * 128;
    if (m < p.M && n < p.N) tile<4, 4>(p, smem, m, p.M, n, static_cast<const bf16_t*>(p.W));
    return;
  }
  int m0 = mt * kTile, m_end = p.M, expert = 0;
  if (p.tiles) {
    expert = p.tiles[2 * mt];
    if (expert < 0) return;
    m0 = p.tiles[2 * mt + 1];
    m_end = min(p.offsets[expert + 1], m0 + kTile);
  }
  tile<8, 2>(p, smem, m0, m_end, n0, static_cast<const bf16_t*>(p.W) + (long)expert * p.N * p.K);
}

void launch_gemm_wide(const GemmArgs& a, hipStream_t s) {
  const int tiles = (a.tiles ? a.n_tiles : (a.M + kTile - 1) / kTile) * ((a.N + kTile - 1) / kTile), left = tiles % 256;
  const int whole = !a.tiles && tiles > 256 && left <= 128 ? tiles - left : tiles;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_wide_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  gemm_wide_kernel<<<whole + 4 * (tiles - whole), 256, kLds, s>>>(a, whole);
  SHAI_CHECK_LAUNCH();
}

}  // namespace shai_lm
