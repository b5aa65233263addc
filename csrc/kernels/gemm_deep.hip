// The LDS-DMA GEMM / convolution of gemm_lds.hip for problems that leave the chip idle: few rows (one image of a classifier, the
// deep levels of a batch-1 UNet, a text encoder, a short prompt), or widths that 256-row tiles do not fill.
//
// What bounds them is the chain of one K-tile: DMA latency with one tile in flight, then wait, barrier, fragment reads and
// dependent MFMAs of a single wave per SIMD (0.6 us per 64 k at the 128 x 64 tile; 197 rows x 768 columns, K = 768 are 24 such
// workgroups).  So:
//   64 x 64, two groups of four waves that take half of every K-tile's MFMA steps each (two waves per SIMD, half the chain),
//     3 tiles in flight, four times the workgroups of 128 x 128.  Four groups were slower (the join costs more than it saves),
//     8 stages too (one workgroup per CU instead of two).
//   128 x 64 in the same form, 2 tiles in flight: 512 .. 8192 rows.
//   128 x 128, eight waves, 3 tiles in flight: K from 1024 on with some thousand rows.
// Replays of a HIP graph over weights that rotate, us per GEMM with its fold (before: the best tile of gemm_lds.hip with its best
// split of K; M x N x K): 197 x 768 x 768 8.4 -> 6.2, 197 x 3072 x 768 12.3 -> 6.8, 197 x 768 x 3072 12.4 -> 10.3 (4 splits),
// 154 x 4096 x 1024 13.7 -> 7.6, 512 x 1280 x 1280 14.4 -> 8.5, 2048 x 640 x 2560 22.7 -> 17.9, 8192 x 320 x 1280 19.4 -> 17.6
// (128 x 128: 14.3), 4096 x 1024 x 2816 35.1 -> 29.9.  Which one runs is the autotuner's choice, like that of every tile.
//   192 x 128, two groups along K of four waves (96 x 64 each), 3 tiles in flight: a row count between, one round of the chip where
//     128 x 128 takes two (6304 x 768 x 3072: 198 workgroups of 300) and, as K is split inside the workgroup, without a fold:
//     47.2 -> 37.2, 4096 x 1280 x 5120 74.5 (256 x 320, four parts) -> 58.5, 512 x 9216 x 3072 56.2 -> 41.4, a convolution of 512 x
//     1280 x 23040 63.0 -> 49.6.  Its sums meet in two passes: all of them are larger than the ring.
//   128 x 128 in that form: LDS gives 64 KB of fragments per K-tile instead of 96.  4096 x 1024 x 2816 28.5 -> 27.9, 1024 x 3072 x 12288
//     100.2 (256 x 256, four parts) -> 83.5.
//   192 x 128, four waves, 1 tile in flight, two workgroups to a CU: the end of one beside the other's loop.  1024 x 9216 x 3072 83.6 ->
//     74.0, 3700 x 5632 x 1024 gated 60.4 -> 56.6, 16384 x 640 x 2560 65.9 -> 64.0.
// Their LDS DMA runs at half the 118 to 130 GB/s a CU that it reaches alone (any pitch, one line or eight an instruction): what bounds
// them is the MFMA pipe (52 % busy), a third of the waves' time at the barrier or waiting for loads.
// (The first two with 8-byte stores; 16-byte ones, gemm_lds_kernel.h, take about a tenth off either.)
// (Operands straight into registers, with the waves splitting K, were tried too: 16 rows x 64 bytes per load instruction reach
// 14 bytes per clock and CU, LDS-DMA 30.)
#include "gemm_lds_kernel.h"

#include <type_traits>

namespace shai {

namespace {

// Tile, waves (rows x columns x groups along K), K-tiles in the ring.
struct Deep {
  int bm, bn, wm, wn, wk, stages;
};
constexpr Deep kDeep[kDeepCfgs] = {{64, 64, 2, 2, 2, 4}, {128, 64, 2, 2, 2, 3}, {128, 128, 2, 4, 1, 4},
                                   {192, 128, 2, 2, 2, 4}, {128, 128, 2, 2, 2, 4}, {192, 128, 2, 2, 1, 2}};

template <int W, bool CONV, bool GLU, int ACT, bool SPLITK>
void launch_one(const GemmArgs& a, float* ws, int splits, int kps, hipStream_t s) {
  constexpr Deep D = kDeep[W];
  constexpr int BM = D.bm, BN = D.bn, ST = D.stages;
  const int tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  constexpr size_t lds = (size_t)ST * (BM + BN) * BK2 * sizeof(bf16_t);
  static_assert(lds <= 160 * 1024, "ring larger than a CU's LDS");
  const dim3 grid(tiles, SPLITK ? splits : (a.batch > 0 ? a.batch : 1));
  auto run = [&](auto epi) {
    gemm2_kernel<BM, BN, D.wm, D.wn, CONV, CONV, GLU, ACT, SPLITK, ST, D.wk, decltype(epi)::value>
        <<<grid, D.wm * D.wn * D.wk * 64, lds, s>>>(a, ws, kps, nullptr);
  };
#define SHAI_EPI(E) run(std::integral_constant<int, E>())
  if constexpr (SPLITK) {
    SHAI_EPI(0);
  } else {
    const bool eight = epilogue8_fits<GLU>(a);
    if constexpr (!CONV) {
      if (a.row_mr != nullptr) return eight ? SHAI_EPI(kEpi8 | kEpiLn) : SHAI_EPI(kEpiLn);
    }
    eight ? SHAI_EPI(kEpi8) : SHAI_EPI(0);
  }
#undef SHAI_EPI
}

template <int W, bool CONV>
void launch_tile(const GemmArgs& a, float* ws, int splits, hipStream_t s) {
  const int kt = (a.K + BK2 - 1) / BK2, kps = (kt + splits - 1) / splits * BK2;
  if (splits > 1) {
    launch_one<W, CONV, false, ACT_NONE, true>(a, ws, splits, kps, s);
    if (!a.no_fold) launch_splitk_epilogue(a, ws, splits, s);
    return;
  }
#define SHAI_DEEP(GLU_, ACT_) launch_one<W, CONV, GLU_, ACT_, false>(a, nullptr, 1, kps, s)
  if constexpr (CONV) {
    if (a.act == ACT_SILU) SHAI_DEEP(false, ACT_SILU);
    else SHAI_DEEP(false, ACT_NONE);
  } else if (a.glu) {
    if (a.act == ACT_SILU) SHAI_DEEP(true, ACT_SILU);
    else if (a.act == ACT_GELU_TANH) SHAI_DEEP(true, ACT_GELU_TANH);
    else SHAI_DEEP(true, ACT_GELU);
  } else {
    switch (a.act) {
      case ACT_SILU: SHAI_DEEP(false, ACT_SILU); break;
      case ACT_GELU: SHAI_DEEP(false, ACT_GELU); break;
      case ACT_GELU_TANH: SHAI_DEEP(false, ACT_GELU_TANH); break;
      case ACT_QUICK_GELU: SHAI_DEEP(false, ACT_QUICK_GELU); break;
      case ACT_RELU: SHAI_DEEP(false, ACT_RELU); break;
      default: SHAI_DEEP(false, ACT_NONE); break;
    }
  }
#undef SHAI_DEEP
}

template <bool CONV>
void launch_which(const GemmArgs& a, int which, float* ws, int splits, hipStream_t s) {
  switch (which) {
    case 0: launch_tile<0, CONV>(a, ws, splits, s); break;
    case 1: launch_tile<1, CONV>(a, ws, splits, s); break;
    case 2: launch_tile<2, CONV>(a, ws, splits, s); break;
    case 3: launch_tile<3, CONV>(a, ws, splits, s); break;
    case 4: launch_tile<4, CONV>(a, ws, splits, s); break;
    default: launch_tile<5, CONV>(a, ws, splits, s); break;
  }
}

}  // namespace

bool gemm_deep_supported(const GemmArgs& a) {
  if (a.rms || a.w_scale || a.w_slice_rows || a.in_scale || a.upsample == 2) return false;
  if (a.row_mr && (a.conv || a.batch > 1)) return false;
  // a convolution's K-tile lies in one filter tap and one source
  return !a.conv || (a.Cin % 64 == 0 && (a.A2 == nullptr || a.Cin1 % 64 == 0));
}

int gemm_deep_wave_groups(int which) { return kDeep[which].wk; }

void gemm_deep_tile(int which, int* bm, int* bn) {
  *bm = kDeep[which].bm;
  *bn = kDeep[which].bn;
}

void launch_gemm_deep(const GemmArgs& a, int which, float* ws, int splits, hipStream_t s) {
  if (ws == nullptr) splits = 1;
  if (a.conv) launch_which<true>(a, which, ws, splits, s);
  else launch_which<false>(a, which, ws, splits, s);
}

}  // namespace shai
