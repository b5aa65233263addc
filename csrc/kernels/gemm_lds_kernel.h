// The kernel of gemm_lds.hip (its comment says how it works) and gemm_deep.hip: LDS-DMA GEMM / implicit-GEMM convolution with
// STAGES K-tiles in LDS.
#pragma once
#include "common.h"
#include "launchers.h"
#include "gemm_epilogue.h"

namespace shai {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int BK2 = 64;
constexpr uint32_t OOB = 0x80000000u;

__device__ __forceinline__ int swz2(int row, int ch) { return row * BK2 + ((ch ^ ((row >> 1) & 7)) << 3); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ void glds16(__amdgpu_buffer_rsrc_t r, bf16_t* lds_wave_base, uint32_t voff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)lds_wave_base, 16, voff, 0, 0, 0);
}

// Epilogue of an unsplit kernel: 8 columns a lane (epilogue8) instead of 4, and a folded LayerNorm.  Kernels of their own: all of it in
// one costs the large tiles their registers (256 x 320: 220, in one kernel 256 and spills, 8192 x 4096 x 4096 330 -> 1790 us) and
// widths that 16 bytes do not fit a tenth (8192 x 330 x 1024 at 128 x 128: 37.5 -> 40.8).
enum { kEpi8 = 1, kEpiLn = 2 };

// WK > 1: that many groups of WM x WN waves, each taking 4 / WK of a K-tile's MFMA steps of the whole tile.
template <int BM, int BN, int WM, int WN, bool CONV, bool FAST, bool GLU, int ACT, bool SPLITK, int STAGES, int WK = 1, int EPI = 0>
__global__ void __launch_bounds__(WM * WN * WK * 64) gemm2_kernel(const GemmArgs p, float* __restrict__ ws, int k_per_split,
                                                             unsigned* __restrict__ cnt) {
  constexpr int NW = WM * WN * WK;
  constexpr int NT = NW * 64;
  constexpr int TM = BM / WM, TN = BN / WN;     // wave tile
  constexpr int IM = TM / 32, JN = TN / 32;     // 32x32 blocks per wave
  constexpr int JA = BM / 8 / NW;               // A wave-instructions per K tile
  constexpr int JB = BN / 8 / NW;               // W wave-instructions per K tile
  static_assert(JA >= 1 && JB >= 1 && IM >= 1 && JN >= 1, "bad tile config");
  constexpr int STAGE = (BM + BN) * BK2;        // elements per stage
  extern __shared__ __attribute__((aligned(16))) bf16_t smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wid / (WM * WN), wm = wid / WN % WM, wn = wid % WN;

  // ---- tile mapping (XCD remap + grouped M ordering)
  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  int bid = blockIdx.x;
  {
    const int xcd = bid & 7, q = total >> 3, r = total & 7;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (bid >> 3);
  }
  constexpr int GROUP = 8;
  const int group = bid / (GROUP * tiles_n);
  const int first_m = group * GROUP;
  const int gsize = min(tiles_m - first_m, GROUP);
  const int in_group = bid - group * GROUP * tiles_n;
  const int m0 = (first_m + in_group % gsize) * BM;
  const int n0 = (in_group / gsize) * BN;
  const int b = SPLITK ? 0 : blockIdx.y;
  const int kz = SPLITK ? blockIdx.y : 0;
  const int k_begin = kz * k_per_split;
  const int k_end = min(p.K, k_begin + k_per_split);

  const bf16_t* A = p.A + (long)b * p.batch_a;
  const bf16_t* Wt = p.W + (long)b * p.batch_w;

  // ---- buffer descriptors (range check = zero fill)
  const __amdgpu_buffer_rsrc_t rW = make_rsrc(Wt, (uint32_t)min((long)p.N * p.ldw * 2, 0x7fffffffL));
  __amdgpu_buffer_rsrc_t rA, rA2;
  if constexpr (CONV) {
    rA = make_rsrc(A, (uint32_t)min((long)p.Nimg * p.H * p.Wd * (p.A2 ? p.Cin1 : p.Cin) * 2, 0x7fffffffL));
    rA2 = p.A2 ? make_rsrc(p.A2, (uint32_t)min((long)p.Nimg * p.H * p.Wd * (p.Cin - p.Cin1) * 2, 0x7fffffffL))
               : rA;
  } else {
    rA = make_rsrc(A, (uint32_t)min((long)p.M * p.lda * 2, 0x7fffffffL));
    rA2 = rA;
  }

  // ---- per-lane staging geometry
  const int lrow = lane >> 3;      // row within an 8-row wave instruction
  const int lpos = lane & 7;       // LDS chunk position
  int a_row[JA], a_ch[JA];
  int cn[JA], coh[JA], cow[JA];
  bool cvalid[JA];
#pragma unroll
  for (int j = 0; j < JA; ++j) {
    const int r = (wid * JA + j) * 8 + lrow;
    a_row[j] = r;
    a_ch[j] = lpos ^ ((r >> 1) & 7);
    if constexpr (CONV) {
      const int m = m0 + r;
      cvalid[j] = m < p.M;
      const int mm = cvalid[j] ? m : 0;
      const int hw = p.OH * p.OW;
      cn[j] = mm / hw;
      const int rem = mm - cn[j] * hw;
      coh[j] = rem / p.OW;
      cow[j] = rem - coh[j] * p.OW;
    }
  }
  int w_row[JB], w_ch[JB];
#pragma unroll
  for (int j = 0; j < JB; ++j) {
    const int r = (wid * JB + j) * 8 + lrow;
    w_row[j] = r;
    w_ch[j] = lpos ^ ((r >> 1) & 7);
  }

  // Convolution whose K-tiles lie in one filter tap and source, up to 32 taps, no upsampling: an output pixel's taps inside the
  // image are bits of a mask, its source address is linear in the tap, and the tap advances with the K-tiles in scalar registers.
  // A lane's address is an add and a select; the divisions and bounds checks of every tile's addresses took longer than its MFMAs
  // (3 x 3 over 8 x 512 x 512, 128 -> 128 channels, 128 x 128 tile: 888 -> 796 us; eight waves and
  // four stages 1165 -> 930).
  [[maybe_unused]] uint32_t c_taps[JA], c_off[JA], c_off2[JA];
  [[maybe_unused]] int t_c = 0, t_kh = 0, t_kw = 0;
  [[maybe_unused]] bool linear = false;
  if constexpr (CONV && FAST) {
    linear = !p.upsample && p.KH * p.KW <= 32;
    const int tap = k_begin / p.Cin;
    t_c = __builtin_amdgcn_readfirstlane(k_begin - tap * p.Cin);
    t_kh = __builtin_amdgcn_readfirstlane(tap / p.KW);
    t_kw = __builtin_amdgcn_readfirstlane(tap - tap / p.KW * p.KW);
    const int cs = p.A2 ? p.Cin1 : p.Cin;
#pragma unroll
    for (int j = 0; j < JA; ++j) {
      const int ih = coh[j] * p.stride - p.pad, iw = cow[j] * p.stride - p.pad;
      uint32_t cols = 0, taps = 0;
      if (linear && cvalid[j]) {
        for (int kw = 0; kw < p.KW; ++kw) cols |= (uint32_t)((unsigned)(iw + kw) < (unsigned)p.Wd) << kw;
        for (int kh = 0; kh < p.KH; ++kh) taps |= (unsigned)(ih + kh) < (unsigned)p.H ? cols << (kh * p.KW) : 0u;
      }
      const uint32_t pix = (uint32_t)((cn[j] * p.H + ih) * p.Wd + iw);   // before the image for a first tap outside it: mod 2^32
      c_taps[j] = taps;
      c_off[j] = (pix * (uint32_t)cs + a_ch[j] * 8) * 2;
      c_off2[j] = (pix * (uint32_t)(p.Cin - p.Cin1) + a_ch[j] * 8) * 2;
    }
  }

  // calls come in the order of the K-tiles
  auto stage = [&](int buf, int k0) {
    bf16_t* sa = smem + buf * STAGE;
    bf16_t* sw = sa + BM * BK2;
#pragma unroll
    for (int j = 0; j < JB; ++j) {
      const int n = n0 + w_row[j], k = k0 + w_ch[j] * 8;
      const uint32_t off = (n < p.N && k < k_end) ? (uint32_t)(((long)n * p.ldw + k) * 2) : OOB;
      glds16(rW, sw + (wid * JB + j) * 8 * BK2, off);
    }
    if constexpr (!CONV) {
#pragma unroll
      for (int j = 0; j < JA; ++j) {
        const int m = m0 + a_row[j], k = k0 + a_ch[j] * 8;
        const uint32_t off = (m < p.M && k < k_end) ? (uint32_t)(((long)m * p.lda + k) * 2) : OOB;
        glds16(rA, sa + (wid * JA + j) * 8 * BK2, off);
      }
    } else if (FAST && linear) {
      const bool second = p.A2 != nullptr && t_c >= p.Cin1;
      const int cs = p.A2 ? (second ? p.Cin - p.Cin1 : p.Cin1) : p.Cin;
      const uint32_t at = (uint32_t)(((t_kh * p.Wd + t_kw) * cs + t_c - (second ? p.Cin1 : 0)) * 2);
      const uint32_t tap = k0 < k_end ? 1u << (t_kh * p.KW + t_kw) : 0u;
#pragma unroll
      for (int j = 0; j < JA; ++j)
        glds16(second ? rA2 : rA, sa + (wid * JA + j) * 8 * BK2, c_taps[j] & tap ? (second ? c_off2[j] : c_off[j]) + at : OOB);
      t_c += BK2;
      if (t_c >= p.Cin) {
        t_c = 0;
        if (++t_kw == p.KW) t_kw = 0, ++t_kh;
      }
    } else {
      int tapF = 0, c0F = 0;
      bool secondF = false;
      if constexpr (FAST) {
        tapF = k0 / p.Cin;
        c0F = k0 - tapF * p.Cin;
        secondF = p.A2 != nullptr && c0F >= p.Cin1;
      }
#pragma unroll
      for (int j = 0; j < JA; ++j) {
        const int k = k0 + a_ch[j] * 8;
        int tap, c;
        bool second;
        if constexpr (FAST) {
          tap = tapF;
          c = c0F + a_ch[j] * 8;
          second = secondF;
        } else {
          tap = k / p.Cin;
          c = k - tap * p.Cin;
          second = p.A2 != nullptr && c >= p.Cin1;
        }
        const int kh = tap / p.KW, kw = tap - kh * p.KW;
        int ih, iw;
        bool ok = cvalid[j] && k < k_end;
        if (p.upsample) {
          const int uh = coh[j] - p.pad + kh, uw = cow[j] - p.pad + kw;
          ok = ok && uh >= 0 && uh < 2 * p.H && uw >= 0 && uw < 2 * p.Wd;
          ih = uh >> 1;
          iw = uw >> 1;
        } else {
          ih = coh[j] * p.stride - p.pad + kh;
          iw = cow[j] * p.stride - p.pad + kw;
          ok = ok && ih >= 0 && ih < p.H && iw >= 0 && iw < p.Wd;
        }
        const int cs = p.A2 ? (second ? p.Cin - p.Cin1 : p.Cin1) : p.Cin;
        const int cc = second ? c - p.Cin1 : c;
        const uint32_t off = ok ? (uint32_t)(((((long)cn[j] * p.H + ih) * p.Wd + iw) * cs + cc) * 2) : OOB;
        if constexpr (FAST) {
          glds16(secondF ? rA2 : rA, sa + (wid * JA + j) * 8 * BK2, off);
        } else {
          // non-uniform source choice: two masked loads into the same LDS slot are not allowed,
          // so a per-lane selected descriptor is not expressible; the generic path needs A2 == null.
          glds16(rA, sa + (wid * JA + j) * 8 * BK2, off);
        }
      }
    }
  };

  float16_ acc[IM][JN];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int nk = k_end > k_begin ? (k_end - k_begin + BK2 - 1) / BK2 : 0;
  const int fr = lane & 31, fh = lane >> 5;
  // W's fragment rows: in order, or, for 8 columns a lane, with bits 2 and 3 of the row exchanged, so that a lane's register groups 2h
  // and 2h + 1 are the 8 consecutive columns 16h + 8fh of the 32 and one 16-byte store takes them.  8-byte stores, 32 rows by 16 bytes
  // an instruction, were most of a short K's time: 6304 x 3072, K = 64 21.5 -> 14.7 us at the 128 x 64 tile, K = 768 53.4 -> 48.4 (128 x
  // 128: 51.2 -> 44.3), 8192 x 960, K = 320 14.5 -> 12.2, 6304 x 768, K = 768 17.8 -> 15.7.  (Whole lines by way of LDS: 1 .. 3 % more,
  // not worth the second path.)
  const int fw = EPI & kEpi8 ? (fr & 19) | (fr & 4) << 1 | (fr & 8) >> 1 : fr;
  // AHEAD: fragments of the next MFMA step are read beside the MFMAs of this one, across the barrier between K-tiles too.  One after
  // the other, by all waves at once behind each barrier, LDS idled beside the MFMAs and they beside it: us before -> after, 4096 x 1024 x
  // 2816 31.0 -> 28.5 (128 x 128, four stages), 512 x 1280 x 5120 21.3 -> 19.6 (64 x 64), 6304 x 768 x 3072 39.8 -> 36.8 (192 x 128), 2048 x
  // 640 x 2560 37.1 -> 35.5 (128 x 128, two stages).  The 128 x 64 tile of two stages, three to a CU, lost (46.9 -> 49.5); the larger
  // eight-wave ones have no registers for it.
  constexpr bool AHEAD = STAGES > 2 || (WM * WN == 4 && IM * JN >= 4);
  if constexpr (!AHEAD) {
    if (nk > 0) {
      stage(0, k_begin);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
    auto compute = [&](int buf) {
      const bf16_t* sa = smem + buf * STAGE;
      const bf16_t* sw = sa + BM * BK2;
#pragma unroll
      for (int t = 0; t < 4 / WK; ++t) {
        const int s = wk * (4 / WK) + t;
        bf16x8 af[IM], wf[JN];
#pragma unroll
        for (int i = 0; i < IM; ++i) af[i] = *reinterpret_cast<const bf16x8*>(sa + swz2(wm * TM + i * 32 + fr, 2 * s + fh));
#pragma unroll
        for (int j = 0; j < JN; ++j) wf[j] = *reinterpret_cast<const bf16x8*>(sw + swz2(wn * TN + j * 32 + fw, 2 * s + fh));
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
          for (int j = 0; j < JN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[j], af[i], acc[i][j], 0, 0, 0);
      }
    };
    for (int kt = 0; kt < nk; ++kt) {
      const int cur = kt & 1;
      if (kt + 1 < nk) stage(cur ^ 1, k_begin + (kt + 1) * BK2);
      compute(cur);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
    }
  } else {
    // A ring of STAGES tiles.  In the last step of tile t a counted vmcnt retires this wave's DMA of tile t + 1 (FIFO), its reads of
    // tile t have arrived, and a raw s_barrier makes both true of every wave: tile t's buffer takes tile t + STAGES, and tile t + 1
    // is read.  Tiles past the end are issued too (every lane out of range: zeros, no traffic), so that the count before each tile
    // is the same; the last wait drains them.
    constexpr int PER = JA + JB;  // DMA instructions per wave per tile
    constexpr int KS = 4 / WK;
    static_assert((STAGES - 1) * PER < 64, "vmcnt has six bits");
    static_assert(KS % 2 == 0, "two sets of fragments take turns");
    // fragments of this wave group's MFMA step t of the K-tile in buffer buf
    struct Frags {
      bf16x8 a[IM], w[JN];
    };
    auto read = [&](int buf, int t, Frags& f) {
      const bf16_t* sa = smem + buf * STAGE;
      const bf16_t* sw = sa + BM * BK2;
      const int s = wk * (4 / WK) + t;
#pragma unroll
      for (int i = 0; i < IM; ++i) f.a[i] = *reinterpret_cast<const bf16x8*>(sa + swz2(wm * TM + i * 32 + fr, 2 * s + fh));
#pragma unroll
      for (int j = 0; j < JN; ++j) f.w[j] = *reinterpret_cast<const bf16x8*>(sw + swz2(wn * TN + j * 32 + fw, 2 * s + fh));
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[j], f.a[i], acc[i][j], 0, 0, 0);
    };
    Frags x[2];
    auto meet = [] {
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int s = 0; s < STAGES; ++s) stage(s, k_begin + s * BK2);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((STAGES - 1) * PER) : "memory");
    meet();
    read(0, 0, x[0]);
    int buf = 0;
    for (int kt = 0; kt < nk; ++kt) {
      const int next = buf == STAGES - 1 ? 0 : buf + 1;
#pragma unroll
      for (int t = 0; t < KS; ++t) {
        if (t < KS - 1) {
          read(buf, t + 1, x[(t + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
        } else {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((STAGES - 2) * PER) : "memory");
#pragma unroll
          for (int i = 0; i < IM; ++i) asm volatile("" : "+v"(x[t & 1].a[i]));
#pragma unroll
          for (int j = 0; j < JN; ++j) asm volatile("" : "+v"(x[t & 1].w[j]));
          meet();
          read(next, 0, x[(t + 1) & 1]);
          __builtin_amdgcn_sched_barrier(0);
          stage(buf, k_begin + (kt + STAGES) * BK2);
        }
        multiply(x[t & 1]);
      }
      buf = next;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  // ---- epilogue: lane owns row m, 4 groups of 4 consecutive n (2 of 8 with kEpi8) per 32x32 block.  WK > 1: the wave groups' sums meet in
  // LDS (the ring is free by now) and are added in group order; each group finishes 4 / WK of the four column groups.
  if constexpr (WK > 1) {
    constexpr int BLOCKS = IM * JN, PASS = NW * BLOCKS * 4096 <= STAGES * STAGE * 2 ? BLOCKS : BLOCKS / 2;   // blocks of a wave at a time
    static_assert(BLOCKS % PASS == 0 && NW * PASS * 4096 <= STAGES * STAGE * 2, "partial tiles larger than the ring");
    float4_* part = reinterpret_cast<float4_*>(smem);
#pragma unroll
    for (int b0 = 0; b0 < BLOCKS; b0 += PASS) {
      __syncthreads();
#pragma unroll
      for (int b = 0; b < PASS; ++b)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float16_& a = acc[(b0 + b) / JN][(b0 + b) % JN];
          part[((wid * PASS + b) * 4 + g) * 64 + lane] = float4_{a[4 * g], a[4 * g + 1], a[4 * g + 2], a[4 * g + 3]};
        }
      __syncthreads();
#pragma unroll
      for (int b = 0; b < PASS; ++b)
#pragma unroll
        for (int g = 0; g < 4 / WK; ++g) {
          const int at = (wid % (WM * WN) * PASS + b) * 4 + wk * (4 / WK) + g;
          float4_ t[WK];
#pragma unroll
          for (int q = 0; q < WK; ++q) t[q] = part[(at + q * WM * WN * PASS * 4) * 64 + lane];
#pragma unroll
          for (int q = 1; q < WK; ++q) t[0] += t[q];
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[(b0 + b) / JN][(b0 + b) % JN][4 * g + e] = t[0][e];
        }
    }
  }
  constexpr int G1 = 4 / WK;
  const int g0 = wk * G1;
  // In-launch split-K fixup (tiles with <= 4 32x32 blocks per wave; the skinny kernel's write-through hand-off, gemv.hip): every K group
  // stores its fp32 partial tile write-through (sc1), drains, joins the barrier and takes a ticket; the group
  // drawing the last one re-arms it, sums the slabs in K-group order (its own from registers, so the sum matches
  // the separate fold bit for bit whatever the arrival order) and runs the full epilogue.  Batch-1 SD2.1 steps
  // run most of their GEMMs split-K at these tiles: the fold kernel was 8.7 % of their kernel time.
  constexpr bool FIXOK = IM * JN <= 4 && !(BM == 128 && BN == 128) && STAGES <= 3 && WK == 1;
  if constexpr (SPLITK && FIXOK) {
    if (cnt != nullptr) {
      __shared__ unsigned g2_last;
      const int S = gridDim.y;
      const __amdgpu_buffer_rsrc_t rws = make_rsrc(ws, (uint32_t)min((long)S * p.M * p.N * 4, 0x7fffffffL));
#pragma unroll
      for (int i = 0; i < IM; ++i) {
        const int m = m0 + wm * TM + i * 32 + fr;
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int n = n0 + wn * TN + j * 32 + 8 * g + 4 * fh;
            const uint32_t off = (uint32_t)(((long)kz * p.M * p.N + (long)m * p.N + n) * 4);
            if (m < p.M && n + 3 < p.N) {
              const float4_ v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
              __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_, v), rws, (int)off, 0, 16);
            } else if (m < p.M) {
              for (int e = 0; e < 4 && n + e < p.N; ++e)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[i][j][4 * g + e]), rws, (int)(off + 4 * e), 0,
                                                      16);
            }
          }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (tid == 0) {
        const unsigned old = __hip_atomic_fetch_add(&cnt[blockIdx.x], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        g2_last = old == (unsigned)(S - 1);
      }
      __syncthreads();
      if (g2_last == 0u) return;
      if (tid == 0) __hip_atomic_store(&cnt[blockIdx.x], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // slabs in rounds of U: every (i, j, g) group's loads of the round are issued before the first add (a
      // load-add chain per slab and group made the fixup latency-bound); the own slab is re-read and replaced by
      // the registers, so the sum order is the K-group order
      float4_ tot[IM][JN][4];
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
          for (int g = 0; g < 4; ++g) tot[i][j][g] = float4_{0.f, 0.f, 0.f, 0.f};
      constexpr int U = IM * JN <= 2 ? 2 : 1;  // slabs per round (registers: U x the tile's accumulators)
      for (int q0 = 0; q0 < S; q0 += U) {
        float4_ ld[U][IM][JN][4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int q = min(q0 + u, S - 1);
#pragma unroll
          for (int i = 0; i < IM; ++i) {
            const int m = min(m0 + wm * TM + i * 32 + fr, p.M - 1);
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
              for (int g = 0; g < 4; ++g) {
                const int n = min(n0 + wn * TN + j * 32 + 8 * g + 4 * fh, ((p.N - 1) & ~3));
                const uint32_t off = (uint32_t)(((long)q * p.M * p.N + (long)m * p.N + n) * 4);
                ld[u][i][j][g] = __builtin_bit_cast(float4_, __builtin_amdgcn_raw_buffer_load_b128(rws, (int)off, 0, 16));
              }
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int q = q0 + u;
          if (q >= S) continue;
#pragma unroll
          for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
              for (int g = 0; g < 4; ++g) {
                const float4_ own = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                tot[i][j][g] += q == kz ? own : ld[u][i][j][g];
              }
        }
      }
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
          for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][4 * g + e] = tot[i][j][g][e];
      bf16_t* C = p.C;
#pragma unroll
      for (int i = 0; i < IM; ++i) {
        const int m = m0 + wm * TM + i * 32 + fr;
        if (m >= p.M) continue;
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int n = n0 + wn * TN + j * 32 + 8 * g + 4 * fh;
            if (n >= p.N) continue;
            float v[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
            epilogue4<GLU, ACT>(p, C, p.residual, m, n, v, 0);
          }
      }
      return;
    }
  }
  if constexpr (SPLITK) {
    float* W = ws + (long)kz * p.M * p.N;
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      const int m = m0 + wm * TM + i * 32 + fr;
      if (m >= p.M) continue;
#pragma unroll
      for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int g = 0; g < G1; ++g) {
          const int n = n0 + wn * TN + j * 32 + 8 * (g0 + g) + 4 * fh;
          if (n + 3 < p.N) {
            float4_ v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
            *reinterpret_cast<float4_*>(W + (long)m * p.N + n) = v;
          } else {
            for (int e = 0; e < 4 && n + e < p.N; ++e) W[(long)m * p.N + n + e] = acc[i][j][4 * g + e];
          }
        }
    }
  } else {
    bf16_t* C = p.C + (long)b * p.batch_c;
    const bf16_t* R = p.residual ? p.residual + (long)b * p.batch_r : nullptr;
    constexpr int V = EPI & kEpi8 ? 8 : 4;
    static_assert(G1 * 4 % V == 0, "a lane's columns lie in one wave group");
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      const int m = m0 + wm * TM + i * 32 + fr;
      if (m >= p.M) continue;
      [[maybe_unused]] float2 mr;
      if constexpr (EPI & kEpiLn) mr = *reinterpret_cast<const float2*>(p.row_mr + 2 * (long)m);
#pragma unroll
      for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int g = 0; g < G1 * 4 / V; ++g) {
          const int n = n0 + wn * TN + j * 32 + 8 * g0 + 2 * V * g + V * fh;
          if (n >= p.N) continue;
          float v[V];
#pragma unroll
          for (int e = 0; e < V; ++e) v[e] = acc[i][j][V * g + e];
          if constexpr (EPI & kEpiLn) {  // LayerNorm of A folded in: rstd[m] * (acc - mean[m] * s[n]), W carries the gain
#pragma unroll
            for (int q = 0; q < V; q += 4) {
              float4_ s = {0.f, 0.f, 0.f, 0.f};
              if (V == 8 || n + 3 < p.N) s = *reinterpret_cast<const float4_*>(p.col_s + n + q);
              else
                for (int e = 0; e < 4 && n + e < p.N; ++e) s[e] = p.col_s[n + e];
#pragma unroll
              for (int e = 0; e < 4; ++e) v[q + e] = mr.y * fmaf(-mr.x, s[e], v[q + e]);
            }
          }
          if constexpr (V == 8) epilogue8<GLU, ACT>(p, C, R, m, n, v, b);
          else epilogue4<GLU, ACT>(p, C, R, m, n, v, b);
        }
    }
  }
}

}  // namespace shai
