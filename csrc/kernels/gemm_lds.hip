// bf16 MFMA GEMM / implicit-GEMM convolution, v2: LDS-DMA staging.
//
//   C[b,m,n] = gate[(b*M+m)/G, n] * act(alpha * sum_k A[b,m,k] * W[b,n,k] + bias[n] + bias2d[m/R, n])
//              + res_alpha * Res[b,m,n]
//
// (gate: optional AdaLN-Zero gate rows, e.g. Flux gate_msa / gate_mlp per image.)
//
// Operand tiles move global -> LDS with `buffer_load_dwordx4 ... lds` (no VGPR
// round trip, no ds_write).  The buffer descriptor's range check supplies the
// zero fill: out-of-range lanes (M/N/K tails, conv padding taps) point past
// num_records and read 0, so the implicit-GEMM conv gather needs no branches
// around its loads.  The LDS image is lane-linear per wave instruction (8 rows x
// 128 B), so the XOR bank swizzle is applied to the per-lane SOURCE chunk and
// the same XOR on the ds_read_b128 side (guide rule 21).
//
// Tile configs (BM x BN, waves WM x WN, each wave 64 x (BN/WN) of 32x32 MFMA
// blocks), BK = 64, 2 LDS stages, loads for K-tile t+1 issued before the MFMAs
// of tile t, one vmcnt(0)+barrier per K-tile.  Optional split-K writes fp32
// partials that gemm_splitk_reduce folds together with the full epilogue.
// XCD-aware bijective block remap + grouped ordering along M.
#include "common.h"
#include "launchers.h"
#include "gemm_lds_kernel.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace shai {

// Fold split-K fp32 partials and apply the full epilogue; one thread per 4 columns.
template <bool GLU, int ACT>
__global__ void gemm_splitk_reduce(const GemmArgs p, const float* __restrict__ ws, int splits) {
  const int n4 = (p.N + 3) / 4;
  const long total = (long)p.M * n4;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int m = (int)(i / n4);
    const int n = (int)(i - (long)m * n4) * 4;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    if (n + 3 < p.N && (p.N & 3) == 0) {
      // four partial slabs per round with every load issued before the first add (a dependent
      // load-add chain per split made the fold latency-bound: ~5 us for M = 64 decode GEMMs)
      const float* src = ws + (long)m * p.N + n;
      const long slab = (long)p.M * p.N;
      for (int s0 = 0; s0 < splits; s0 += 4) {
        float4_ x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
          x[u] = s0 + u < splits ? *reinterpret_cast<const float4_*>(src + (s0 + u) * slab) : float4_{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          v[0] += x[u][0]; v[1] += x[u][1]; v[2] += x[u][2]; v[3] += x[u][3];
        }
      }
    } else {
      for (int s = 0; s < splits; ++s) {
        const float* src = ws + (long)s * p.M * p.N + (long)m * p.N + n;
        for (int e = 0; e < 4 && n + e < p.N; ++e) v[e] += src[e];
      }
    }
    if (p.rms) {  // folded RMSNorm: per-row sum of squares partials follow the [splits][M][N] block
      const float* ss = ws + (long)splits * p.M * p.N;
      float t = 0.f;
      for (int s = 0; s < splits; ++s) t += ss[(long)s * p.M + m];
      const float r = rsqrtf(t / p.K + p.rms_eps);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= r;
    }
    // phase conv: row m's output pixel (no residual on that path)
    bf16_t* C = p.upsample == 2 ? p.C + (up2_out_row(p, m) - m) * p.ldc : p.C;
    epilogue4<GLU, ACT>(p, C, p.residual, m, n, v);
  }
}

// ---------------------------------------------------------------------------- dispatch
static int g_stages() {
  static int st = [] {
    const char* e = getenv("SHAI_GEMM_STAGES");
    return (e && e[0] == '3') ? 3 : 2;
  }();
  return st;
}

template <int BM, int BN, int WM, int WN, bool CONV, bool FAST, bool GLU, int ACT, bool SPLITK>
static void launch_cfg(const GemmArgs& a, float* ws, int splits, int kps, hipStream_t s, unsigned* cnt) {
  const int tiles = ((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN);
  dim3 grid(tiles, SPLITK ? splits : (a.batch > 0 ? a.batch : 1));
  auto go = [&](auto kernel, int stages) {
    kernel<<<grid, WM * WN * 64, (size_t)stages * (BM + BN) * BK2 * sizeof(bf16_t), s>>>(a, ws, kps, cnt);
  };
  auto run = [&](auto epi) {
    constexpr int E = decltype(epi)::value;
    if constexpr (3 * (BM + BN) * BK2 * sizeof(bf16_t) <= 160 * 1024 && !(E & kEpiLn)) {
      if (g_stages() == 3) return go(gemm2_kernel<BM, BN, WM, WN, CONV, FAST, GLU, ACT, SPLITK, 3, 1, E>, 3);
    }
    go(gemm2_kernel<BM, BN, WM, WN, CONV, FAST, GLU, ACT, SPLITK, 2, 1, E>, 2);
  };
  if constexpr (SPLITK) {
    run(std::integral_constant<int, 0>());
  } else {
    const bool eight = epilogue8_fits<GLU>(a);
    if constexpr (!CONV) {
      if (a.row_mr != nullptr) {
        if (eight) return run(std::integral_constant<int, kEpi8 | kEpiLn>());
        // 10 blocks of accumulators a wave, 4 columns at a time and a GELU spill: 256 x 256 then
        if constexpr (BM * BN / (WM * WN) > 8 * 1024) return launch_cfg<256, 256, 4, 2, CONV, FAST, GLU, ACT, false>(a, ws, splits, kps, s, cnt);
        else return run(std::integral_constant<int, kEpiLn>());
      }
    }
    if (eight) run(std::integral_constant<int, kEpi8>());
    else run(std::integral_constant<int, 0>());
  }
}

// Tile configs: {BM, BN, WM, WN}.  256x320 covers the SD2.1 channel widths
// (320/640/1280/960/2560... are all multiples of 320) with no N waste and a
// 142 FLOP/B operand intensity; 256x256 for LLM / Flux widths.
struct TileCfg {
  int bm, bn;
  float eff;  // relative per-FLOP efficiency used by the planner
};
static const TileCfg kCfgs[] = {{256, 320, 1.00f}, {256, 256, 1.00f}, {256, 128, 0.90f}, {128, 128, 0.75f},
                                {128, 64, 0.55f}};
constexpr int kNumCfgs = 5;
// Config index space: [0, kNumCfgs) this file's tile configs; kNumCfgs + 0..3 the retired pipelined v3 kernel
// (cached choices run on v4); kNumCfgs + 4 / + 5 the 8-phase ping-pong v4 kernel (gemm_8ph.hip) with 256 / 320 wide tiles,
// kNumCfgs + 6 / + 7 the same in its persistent form (next tile's operands prefetched under the epilogue).
constexpr int kV4Cfg = kNumCfgs + 4;
// kV4Cfg + 4 / + 5: the four-wave kernel (gemm_w4.hip) with 256 x 256 / 256 x 192 tiles (128 x 128 / 128 x 96
// wave tiles; plain GEMM, GLU, folded LayerNorm; conv with the former; no split-K).
constexpr int kW4Cfg = kV4Cfg + 4;
// kW4Cfg + 2: the W-stationary low-K kernel (gemm_ws.hip): K = 320, N a multiple of 320, weights resident in VGPRs,
// persistent over M (plain / bias / act / GLU / residual / folded LayerNorm; no split-K).
constexpr int kWsCfg = kW4Cfg + 2;
// kWsCfg + 1 .. + kDeepCfgs: this file's kernel with smaller tiles and more K-tiles in flight (gemm_deep.hip).
constexpr int kDeepCfg = kWsCfg + 1;


template <bool CONV, bool FAST, bool GLU, int ACT>
static void launch_tiles(const GemmArgs& a, int cfg, float* ws, int splits, int kps, hipStream_t s, unsigned* cnt) {
  const bool sk = splits > 1;
#define SHAI_CFG(BM_, BN_, WM_, WN_)                                                   \
  if (sk) launch_cfg<BM_, BN_, WM_, WN_, CONV, FAST, GLU, ACT, true>(a, ws, splits, kps, s, cnt); \
  else launch_cfg<BM_, BN_, WM_, WN_, CONV, FAST, GLU, ACT, false>(a, ws, splits, kps, s, cnt);
  switch (cfg) {
    case 0: SHAI_CFG(256, 320, 4, 2); break;
    case 1: SHAI_CFG(256, 256, 4, 2); break;
    case 2: SHAI_CFG(256, 128, 4, 2); break;
    case 3: SHAI_CFG(128, 128, 2, 2); break;
    default: SHAI_CFG(128, 64, 2, 2); break;
  }
#undef SHAI_CFG
}

template <bool GLU, int ACT>
static void launch_reduce(const GemmArgs& a, const float* ws, int splits, hipStream_t s) {
  const long total = (long)a.M * ((a.N + 3) / 4);
  long blocks = (total + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  gemm_splitk_reduce<GLU, ACT><<<(int)blocks, 256, 0, s>>>(a, ws, splits);
}

// Cost model: rounds of co-resident blocks x padded tile work / config efficiency.
// Blocks/CU from LDS (2 stages); 256 CUs.  Split-K only when the grid is small.
void gemm2_plan(const GemmArgs& a, int* cfg, int* splits) {
  const long M = a.M, N = a.N, K = a.K;
  const int batch = a.batch > 0 ? a.batch : 1;
  static const int forced = [] {
    const char* e = getenv("SHAI_GEMM_CFG");
    return e ? atoi(e) : -1;
  }();
  double best = 1e300;
  int bc = 3, bs = 1;
  const long kt = (K + BK2 - 1) / BK2;
  for (int c = 0; c < kNumCfgs; ++c) {
    if (forced >= 0 && c != forced) continue;
    const TileCfg& t = kCfgs[c];
    if (a.glu && (t.bn % 4)) continue;
    const long tm = (M + t.bm - 1) / t.bm, tn = (N + t.bn - 1) / t.bn;
    const long tiles = tm * tn * batch;
    const long lds = 2L * (t.bm + t.bn) * BK2 * 2;
    const long per_cu = std::max(1L, std::min(163840L / lds, 2048L / ((t.bm / 64) * (t.bn / 64) * 64 > 512 ? 512 : 256)));
    for (int sp = 1; sp <= 16; sp *= 2) {   // (the tuner's counts made this model choose worse: 1.7 % over 204 problems)
      if (sp > 1 && (batch != 1 || kt / sp < 4)) break;
      const long blocks = tiles * sp;
      const long slots = 256 * per_cu;
      const long rounds = (blocks + slots - 1) / slots;
      const double work = (double)t.bm * t.bn * ((kt + sp - 1) / sp);
      double cost = rounds * work / t.eff;
      if (blocks < slots) cost *= 1.0 + 0.35 * (1.0 - (double)blocks / slots);  // idle CUs still cost latency
      if (sp > 1) cost += 0.02 * work * sp;                                   // partials + reduce pass
      if (cost < best) {
        best = cost;
        bc = c;
        bs = sp;
      }
    }
  }
  *cfg = bc;
  *splits = bs;
  // v4 (8-phase ping-pong) outruns every v2 tile on problems that fill the chip with 256-row tiles
  if (forced < 0 && gemm4_supported(a) && bs == 1) {
    const int bn = (N % 320 == 0 && N % 256 != 0) ? 320 : 256;
    const long tiles = ((M + 255) / 256) * ((N + bn - 1) / bn) * batch;
    if (tiles >= 192 && K >= 256) *cfg = kV4Cfg + (bn == 320 ? 1 : 0);
  }
}

size_t gemm2_workspace_bytes(const GemmArgs& a) {
  int cfg, splits;
  gemm2_plan(a, &cfg, &splits);
  return splits > 1 ? (size_t)splits * a.M * a.N * sizeof(float) : 0;
}

template <bool CONV, bool FAST>
static void launch_all(const GemmArgs& a, float* ws, int cfg, int splits, hipStream_t s) {
  if (ws == nullptr) splits = 1;
  const long kt = (a.K + BK2 - 1) / BK2;
  const int kps = (int)(((kt + splits - 1) / splits) * BK2);
  // split-K at the 256 x 128 / 128 x 64 tiles (cfg 2 / 4): fixed up inside the launch when a ticket slice is available
  // (SHAI_G2_FIXUP=0: the separate fold kernel)
  // Off by default: measured SLOWER end to end (SD2.1 bs1 p50 406 ms with it vs 356 ms with the fold kernel,
  // profiles/norm_handoff_round4.md): the write-through slabs and the last arriver's serial sum cost more than
  // the fold launch they replace.  SHAI_G2_FIXUP=1 enables it (tests force it through the forced-split hook).
  static const bool fixup_on = [] {
    const char* e = getenv("SHAI_G2_FIXUP");
    return e && e[0] == '1';
  }();
  unsigned* cnt = nullptr;
  // (not at 128 x 128: the fixup's registers would halve that config's occupancy)
  if (splits > 1 && (cfg == 2 || cfg == 4) && fixup_on && !a.rms && !a.no_fold && (long)splits * a.M * a.N * 4 < 0x7fffffffL) {
    const int bm = cfg == 2 ? 256 : 128, bn = cfg == 4 ? 64 : 128;
    const long tiles = (long)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
    if (tiles <= 4096) cnt = skinny_ticket_slice(s, (int)tiles);
  }
#define SHAI_G2(GLU_, ACT_)                                                   \
  do {                                                                        \
    launch_tiles<CONV, FAST, GLU_, ACT_>(a, cfg, ws, splits, kps, s, cnt);    \
    if (splits > 1 && cnt == nullptr && !a.no_fold) launch_reduce<GLU_, ACT_>(a, ws, splits, s); \
  } while (0)
  if constexpr (CONV) {  // convs: no GLU, activation none / silu
    if (a.act == ACT_SILU) SHAI_G2(false, ACT_SILU);
    else SHAI_G2(false, ACT_NONE);
  } else if (a.glu) {
    if (a.act == ACT_SILU) SHAI_G2(true, ACT_SILU);
    else if (a.act == ACT_GELU_TANH) SHAI_G2(true, ACT_GELU_TANH);
    else SHAI_G2(true, ACT_GELU);
  } else {
    switch (a.act) {
      case ACT_SILU: SHAI_G2(false, ACT_SILU); break;
      case ACT_GELU: SHAI_G2(false, ACT_GELU); break;
      case ACT_GELU_TANH: SHAI_G2(false, ACT_GELU_TANH); break;
      case ACT_QUICK_GELU: SHAI_G2(false, ACT_QUICK_GELU); break;
      case ACT_RELU: SHAI_G2(false, ACT_RELU); break;
      default: SHAI_G2(false, ACT_NONE); break;
    }
  }
#undef SHAI_G2
}

void launch_gemm2_cfg(const GemmArgs& a, float* ws, int cfg, int splits, hipStream_t s) {
  if (cfg >= kDeepCfg) {
    launch_gemm_deep(a, cfg - kDeepCfg, ws, splits, s);
    return;
  }
  if (cfg == kWsCfg) {  // whole K resident: a split-K choice is run unsplit
    launch_gemm_ws(a, s);
    return;
  }
  if (cfg == kW4Cfg || cfg == kW4Cfg + 1) {  // whole K per tile: a split-K choice is run unsplit
    launch_gemm_w4(a, cfg == kW4Cfg ? 256 : 192, s);
    return;
  }
  if (cfg >= kV4Cfg) {
    const int v = cfg - kV4Cfg;
    launch_gemm4(a, ws, splits, (v & 1) ? 320 : 256, s, v >= 2);
    return;
  }
  if (cfg >= kNumCfgs) {  // retired v3 (pipelined 256x256 / 256x320): a cached choice runs on v4, same tile width
    launch_gemm4(a, ws, splits, cfg - kNumCfgs >= 2 ? 320 : 256, s, false);
    return;
  }
  if (!a.conv) {
    launch_all<false, false>(a, ws, cfg, splits, s);
  } else {
    const bool fast = (a.Cin % 64) == 0 && (a.A2 == nullptr || (a.Cin1 % 64) == 0);
    if (fast) launch_all<true, true>(a, ws, cfg, splits, s);
    else launch_all<true, false>(a, ws, cfg, splits, s);
  }
}

// Split-K fold + full epilogue for fp32 partials laid out [splits][M][N] (also used by the skinny kernel).
void launch_splitk_epilogue(const GemmArgs& a, const float* ws, int splits, hipStream_t s) {
  if (a.glu) {  // every activation: the skinny kernels (any GLU activation) fold through here too
    switch (a.act) {
      case ACT_SILU: launch_reduce<true, ACT_SILU>(a, ws, splits, s); break;
      case ACT_GELU: launch_reduce<true, ACT_GELU>(a, ws, splits, s); break;
      case ACT_GELU_TANH: launch_reduce<true, ACT_GELU_TANH>(a, ws, splits, s); break;
      case ACT_QUICK_GELU: launch_reduce<true, ACT_QUICK_GELU>(a, ws, splits, s); break;
      case ACT_RELU: launch_reduce<true, ACT_RELU>(a, ws, splits, s); break;
      default: launch_reduce<true, ACT_NONE>(a, ws, splits, s); break;
    }
    return;
  }
  switch (a.act) {
    case ACT_SILU: launch_reduce<false, ACT_SILU>(a, ws, splits, s); break;
    case ACT_GELU: launch_reduce<false, ACT_GELU>(a, ws, splits, s); break;
    case ACT_GELU_TANH: launch_reduce<false, ACT_GELU_TANH>(a, ws, splits, s); break;
    case ACT_QUICK_GELU: launch_reduce<false, ACT_QUICK_GELU>(a, ws, splits, s); break;
    case ACT_RELU: launch_reduce<false, ACT_RELU>(a, ws, splits, s); break;
    default: launch_reduce<false, ACT_NONE>(a, ws, splits, s); break;
  }
}

int gemm2_num_cfgs() { return kDeepCfg + kDeepCfgs; }

// Configs the autotuner races: not the retired v3 indices (kNumCfgs .. + 3; the pipelined kernel held 2 cached
// shapes when it was removed -- every index stays valid for old caches).
bool gemm2_cfg_candidate(int cfg) { return !(cfg >= kNumCfgs && cfg < kV4Cfg); }

bool gemm2_cfg_splittable(int cfg) { return cfg != kW4Cfg && cfg != kW4Cfg + 1 && cfg != kWsCfg; }

// One count from each of 2 to 3, 4 to 6, 7 to 12 and 13 to 16: the one with which the tiles' parts leave the fewest of the 256 CUs without one
// in the last round. Workgroups of small tiles share a CU, but where every CU has as many of them none waits: counted by the places that a CU's
// LDS has for them, 4096 columns of 110 rows lost the 256 workgroups of 64 x 64 tiles in two parts to 384 in three, of which half the CUs had
// two (K = 4096, cold weights: 16.9 and 20.9 us with what was taken in their stead).
// Times of what is picked over the best of all counts to 16, in the mean and at most, for 322 convolutions of requests of 320 x 256 to 768 x 768
// pixels and of small batches: 2, 4, 8 and 16, as many launches to time, 1.019 and 1.24, 69 of them over 1.03; by places in LDS 1.0017 and 1.09, 7;
// by CUs 1.0007 and 1.05, 2. For 78 plain products of 70 to 600 rows 1.0025 and 1.09, 1.0020 and 1.04, 1.0007 and 1.03. No part is empty or
// under 4 k-tiles.
int gemm2_split_counts(int M, int N, int K, int cfg, int most, int* out) {
  int bm, bn;
  if (cfg >= kDeepCfg) {
    gemm_deep_tile(cfg - kDeepCfg, &bm, &bn);
  } else if (cfg >= kNumCfgs) {
    bm = 256, bn = cfg >= kV4Cfg && ((cfg - kV4Cfg) & 1) ? 320 : 256;
  } else {
    bm = kCfgs[cfg].bm, bn = kCfgs[cfg].bn;
  }
  const long tiles = (long)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  const int kt = (K + BK2 - 1) / BK2;
  int n = 0;
  out[n++] = 1;
  for (int p = 2; p <= most && p <= 16; p *= 2) {
    int best = 0;
    long best_left = 0, best_rounds = 1;
    for (int s = (4 * p + 4) / 5; 5 * s < 8 * p && s <= 16; ++s) {
      const int per = (kt + s - 1) / s;
      if (kt / s < 4 || (kt + per - 1) / per != s) continue;
      const long rounds = (tiles * s + 255) / 256, left = rounds * 256 - tiles * s;
      if (best == 0 || left * best_rounds < best_left * rounds) best = s, best_left = left, best_rounds = rounds;
    }
    if (best) out[n++] = best;
  }
  return n;
}

bool gemm2_cfg_supported(const GemmArgs& a, int cfg) {
  // an epilogue activation no tile kernel instantiates is never accepted (it would run as another one)
  if (!tile_act_supported(a)) return false;
  // phase-decomposed upsample conv (upsample == 2) / weight slices: only the v4 kernel maps rows to output pixels
  // and tiles to weight slices
  if (a.upsample == 2 || a.w_slice_rows != 0) return cfg >= kV4Cfg && cfg < kV4Cfg + 4 && gemm4_supported(a);
  // folded LayerNorm (row_mr): applied by the unsplit epilogues of this file's tiles (plain GEMMs) and of the v4, the 192-wide four-wave
  // and the W-stationary kernel, batch 1.  The small tiles: 6304 x 2304 x 768 37.6 us (256 x 256) instead of v4's 44.9.
  if (a.row_mr != nullptr) {
    if (cfg == kWsCfg) return gemm_ws_supported(a);
    if (a.batch > 1 || (cfg >= kNumCfgs && cfg < kV4Cfg) || cfg == kW4Cfg) return false;
    if (cfg >= kV4Cfg && cfg < kV4Cfg + 4) return gemm4_supported(a);
    if (a.conv || a.in_scale != nullptr) return false;
  }
  // 192 x 128 and 128 x 128 with two groups of waves along K: up to 8192 rows.  They fill one round of the chip where other tiles
  // need more or a split (4096 x 1280 x 5120: 57.8 us, two workgroups of 192 x 128 to a CU 74.4).  With more rows the better of the two
  // is ahead of the best other tile by 5 % at most (9364 x 512 x 1024 19.6 and 20.6 us, 8274 x 1280 x 5120 115.7 and 116.2) and
  // mostly behind it (9364 x 768 x 768 23.2 and 19.9, 12288 x 1280 x 5120 172 and 132, 16384 x 1024 x 2816 108 and 80).
  if ((cfg == kDeepCfg + 3 || cfg == kDeepCfg + 4) && a.M > 8192) return false;
  if (cfg >= kDeepCfg)
    return cfg < kDeepCfg + kDeepCfgs && gemm_deep_supported(a) && !(keeps_order(a) && gemm_deep_wave_groups(cfg - kDeepCfg) > 1);
  if (cfg == kWsCfg) return gemm_ws_supported(a);
  if (cfg == kW4Cfg) return gemm_w4_supported(a);
  if (cfg == kW4Cfg + 1) return !a.conv && gemm_w4_supported(a);
  if (cfg >= kV4Cfg) return cfg < kV4Cfg + 4 && gemm4_supported(a);
  if (cfg >= kNumCfgs) return gemm4_supported(a);  // retired v3 -> v4
  if (a.in_scale != nullptr) return false;
  if (a.conv && a.A2 != nullptr && (a.Cin % 64 != 0 || a.Cin1 % 64 != 0)) return false;  // 64-wide K tiles
  return cfg >= 0 && cfg < kNumCfgs;
}

void gemm2_cfg_info(int cfg, int* bm, int* bn) {
  if (cfg >= kDeepCfg) {
    gemm_deep_tile(cfg - kDeepCfg, bm, bn);
    return;
  }
  if (cfg == kWsCfg) {  // W-stationary kernel: reported as "1x-320"
    *bm = 1;
    *bn = -320;
    return;
  }
  if (cfg == kW4Cfg || cfg == kW4Cfg + 1) {  // four-wave kernel: reported as "4x-256" / "4x-192"
    *bm = 4;
    *bn = cfg == kW4Cfg ? -256 : -192;
    return;
  }
  if (cfg >= kV4Cfg) {  // 8-phase v4 kernel: reported as "8x-<BN>" ("9x-<BN>" persistent)
    *bm = cfg >= kV4Cfg + 2 ? 9 : 8;
    *bn = ((cfg - kV4Cfg) & 1) ? -320 : -256;
    return;
  }
  if (cfg >= kNumCfgs) {  // retired v3: runs as v4
    *bm = 8;
    *bn = cfg - kNumCfgs >= 2 ? -320 : -256;
    return;
  }
  *bm = kCfgs[cfg].bm;
  *bn = kCfgs[cfg].bn;
}

void launch_gemm2(const GemmArgs& a, float* ws, hipStream_t s) {
  int cfg, splits;
  gemm2_plan(a, &cfg, &splits);
  launch_gemm2_cfg(a, ws, cfg, splits, s);
}

}  // namespace shai
