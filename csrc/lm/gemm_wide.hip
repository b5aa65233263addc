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

#include <algorithm>
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

struct Place {
  int m0, n0;
};

// Tiles one after the other, the next one's first two k-tiles fetched during the last two of the one before: no launch, no first loads to
// wait for, and the stores go out beside the next products (the first wait counts them, as they are younger than what it waits for).  A
// register kept over both halves of an epilogue would spill: one path of stores, no branches in it.  Rows and columns take 16-byte stores, K is at least two k-tiles, no rows are
// gathered.  next(Place&) gives the workgroup's next tile, false: none.
template <typename Next>
__device__ __forceinline__ void chain(const GemmArgs& p, bf16_t* smem, Place at, Next next) {
  constexpr int NB = 8, B = kTile, FR = 2 * NB, STAGE = 2 * B * 64, NQ = NB / 2;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wid >> 1, wn = wid & 1;
  const __amdgpu_buffer_rsrc_t rW = rsrc(p.W, (long)p.N * p.K * 2), rA = rsrc(p.A, ((long)(p.a_rows - 1) * p.lda + p.K) * 2);

  // byte offset of this lane's 16-byte chunk of the NB + NB row groups its wave stages, at k = 0; the bank swizzle is on the source.
  // W's rows are permuted inside pairs of blocks of 16, so that a lane's results are 8 neighbouring columns.
  const int lrow = lane >> 3, lpos = lane & 7;
  uint32_t off[FR];
  auto place = [&](const Place& t, bool any) {
    int lr = lrow, lp = lpos;
    asm volatile("" : "+v"(lr), "+v"(lp));
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int r = wid * (B / 4) + j * 8 + lr, ch = (lp ^ ((r >> 1) & 7)) * 8, m = t.m0 + r;
      const int wave = r / (B / 2), l = r % (B / 2), n = t.n0 + wave * (B / 2) + (l >> 5) * 32 + ((l & 15) >> 2) * 8 + ((l >> 4) & 1) * 4 + (l & 3);
      off[j] = any && m < p.M ? (uint32_t)(((long)m * p.lda + ch) * 2) : kOob;
      off[NB + j] = any && n < p.N ? (uint32_t)(((long)n * p.K + ch) * 2) : kOob;
    }
  };
  const int nk = p.K / 64;
  int base = 0;                                  // the tile's first k-tile in the sequence of all, which the stages follow
  // row group g of the place's k-tile k into the stage of the tile's k-tile t
  auto dma = [&](int t, int k, int g) {
    bf16_t* dst = smem + ((base + t) & 1) * STAGE + ((g < NB ? 0 : B) + wid * (B / 4) + (g % NB) * 8) * 64;
    dma16(g < NB ? rA : rW, dst, off[g] + (uint32_t)k * 128u);
  };
  // fragment f of k-step s: W's blocks of 16 rows first, the first MFMAs need all of them
  const int fr = lane & 15, fq = lane >> 4;
  typedef bf16x8 Set[FR];
  auto read = [&](int t, int s, int f, Set& x) {
    const int row = f < NB ? B + wn * (B / 2) + 16 * f : wm * (B / 2) + 16 * (f - NB);
    x[f] = *reinterpret_cast<const bf16x8*>(smem + ((base + t) & 1) * STAGE + (row + fr) * 64 + (((fq + 4 * s) ^ ((fr >> 1) & 7)) << 3));
  };
  // a set is redefined after its inline wait: the compiler's own wait counts do not see that one
  auto landed = [](Set& x) {
#pragma unroll
    for (int f = 0; f < FR; ++f) asm volatile("" : "+v"(x[f]));
  };

  float4_ acc[NB][NB];
  Set x0, x1;
  place(at, true);
#pragma unroll
  for (int g = 0; g < 2 * FR; ++g) dma(g / FR, g / FR, g % FR);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FR) : "memory");
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
  // k: the place's k-tile that goes into the stage of t + 2; behind: the last tile's stores are younger than the loads waited for
  auto half1 = [&](int t, int k, bool behind) {
    if (behind) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(NB * NQ) : "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    landed(x1);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < NB; ++g) {
      dma(t + 2, k, 2 * g);
      dma(t + 2, k, 2 * g + 1);
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

  bf16_t* C = static_cast<bf16_t*>(p.C);
  for (;;) {
    Place to;
    const bool more = next(to);
    half0(0, std::true_type{});
    for (int t = 0; t + 1 < nk; ++t) {
      if (t == nk - 2) place(to, more);
      half1(t, t + 2 < nk ? t + 2 : t + 2 - nk, base > 0 && t == 0);
      half0(t + 1, std::false_type{});
    }
    half1(nk - 1, 1, false);

    const __amdgpu_buffer_rsrc_t rC = rsrc(C + (long)at.m0 * p.ldc, 0x7fffffffL);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int r = wm * (B / 2) + 16 * i + fr, m = at.m0 + r;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int n = at.n0 + wn * (B / 2) + 32 * q + 8 * fq;
        float4_ u = acc[i][2 * q], v = acc[i][2 * q + 1];
        const bool su = p.epi == EPI_RELU2 && n < p.n_act, sv = p.epi == EPI_RELU2 && n + 4 < p.n_act;   // epilogue_cols without branches
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = fmaxf(u[e], 0.f), y = fmaxf(v[e], 0.f);
          u[e] = su ? x * x : u[e];
          v[e] = sv ? y * y : v[e];
        }
        const uint4_ o = {pack2(u[0], u[1]), pack2(u[2], u[3]), pack2(v[0], v[1]), pack2(v[2], v[3])};
        // always NB * NQ stores: they are counted above
        __builtin_amdgcn_raw_buffer_store_b128(o, rC, m < p.M && n < p.n_main ? ((uint32_t)r * (uint32_t)p.ldc + (uint32_t)n) * 2u : kOob, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!more) return;
    at = to;
    base += nk;
  }
}

}  // namespace

// Workgroups 0 .. step - 1 take tiles step apart of the first `whole`, every four behind them the quarters of one of the remaining tiles.
// The columns of tiles from `lines` on, with side columns, come last: a chain (step < whole) has none.
__global__ void __launch_bounds__(256, 1) gemm_wide_kernel(const GemmArgs p, int whole, int step, int lines) {
  extern __shared__ __attribute__((aligned(16))) bf16_t smem[];
  const int tiles_m = p.tiles ? p.n_tiles : (p.M + kTile - 1) / kTile, tiles_n = (p.N + kTile - 1) / kTile;
  constexpr int GROUP = 8;
  auto tile_of = [&](int bid, int& mt, int& n0) {
    const int first_n = bid < tiles_m * lines ? 0 : lines, cols = first_n ? tiles_n - lines : lines;
    bid -= tiles_m * first_n;
    const int group = bid / (GROUP * cols), first_m = group * GROUP;
    const int gsize = min(tiles_m - first_m, GROUP);
    const int in_group = bid - group * GROUP * cols;
    mt = first_m + in_group % gsize;
    n0 = (first_n + in_group / gsize) * kTile;
  };
  int bid = blockIdx.x, mt, n0;
  if (bid >= step) {
    const int part = (bid - step) & 3;
    tile_of(whole + ((bid - step) >> 2), mt, n0);
    const int m = mt * kTile + (part >> 1) * 128, n = n0 + (part & 1) * 128;
    if (m < p.M && n < p.N) tile<4, 4>(p, smem, m, p.M, n, static_cast<const bf16_t*>(p.W));
    return;
  }
  auto take = [&] {
    const int xcd = bid & 7, q = whole >> 3, r = whole & 7;
    tile_of((xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (bid >> 3), mt, n0);
    bid += step;
  };
  take();
  if (step < whole) {
    chain(p, smem, Place{mt * kTile, n0}, [&](Place& t) {
      if (bid >= whole) return false;
      take();
      t = Place{mt * kTile, n0};
      return true;
    });
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

// Tiles of whole rounds; a last round of up to half of the CUs is cut in quarters.
static int whole_rounds(const GemmArgs& a, int tiles) {
  const int left = tiles % 256;
  return !a.tiles && tiles > 256 && left <= 128 ? tiles - left : tiles;
}

// Tiles that follow each other in their workgroups, 0: every tile has one of its own.  More than a round of tiles without side columns, rows of
// 16-byte stores at 32-bit offsets.  The tiles with side columns are the last and go to quarters, those past the columns exit at once; more than
// an eighth of all are not worth it (4096 x 8192 x 2048 with 2048 side columns 127 -> 133 us).  us: 7700 x 14848 x 2048 414 -> 396, 7700 x 16640
// 465 -> 462, 8192 x 8192 x 8192 837 -> 824; with 32 side columns 7700 x 14624 452 -> 397, 2048 x 14624 122 -> 109, 33000 x 14624 1836 -> 1590; with
// 16, 8192 x 17424 557 -> 480, 7700 x 17424 500 -> 466; one round is the slower through the direct stores (7700 x 2048 x 10496: 262 and 269).
int gemm_wide_chained(const GemmArgs& a) {
  const int tiles_m = (a.M + kTile - 1) / kTile, tiles_n = (a.N + kTile - 1) / kTile;
  const int rounds = whole_rounds(a, tiles_m * tiles_n), lines = a.n_main == a.N ? tiles_n : a.n_main / kTile;
  const int n = std::min(rounds, tiles_m * lines);
  const bool fits = !a.tiles && !a.gather && a.K >= 128 && a.ldc % 8 == 0 && a.ldc <= 1 << 21 && a.n_main % 8 == 0;
  return fits && n > 256 && 8L * n >= 7L * rounds ? n : 0;
}

void launch_gemm_wide(const GemmArgs& a, hipStream_t s) {
  const int tiles_n = (a.N + kTile - 1) / kTile, tiles = (a.tiles ? a.n_tiles : (a.M + kTile - 1) / kTile) * tiles_n;
  const int chained = gemm_wide_chained(a), whole = chained ? chained : whole_rounds(a, tiles), step = chained ? 256 : whole;
  const int lines = chained && a.n_main != a.N ? a.n_main / kTile : tiles_n;
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_wide_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  gemm_wide_kernel<<<step + 4 * (tiles - whole), 256, kLds, s>>>(a, whole, step, lines);
  SHAI_CHECK_LAUNCH();
}

}  // namespace shai_lm
