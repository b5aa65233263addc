// GroupNorm (+ SiLU) of small images in one launch: statistics, normalisation and, behind a split-K convolution, the fold of
// its partial sums.
//
// What bounds a small norm is launches, not bytes: at 4 x 16 x 16 x 1280 the column sums, the finalize and the apply pass took
// 11.2 us in a graph for 5.2 MB, now 5.3 (4 x 8 x 8 x 1280 9.9 -> 3.9, 16 x 16 x 16 x 1280 14.4 -> 8.1, 4 x 32 x 32 x 640 12.0 -> 7.2),
// and the fold of a split convolution is another launch less.  A workgroup owns one image's channels of one group (of two where a
// group's width is no multiple of 4), holds them in registers as bf16, and takes mean and variance in two passes over the registers.
#include "common.h"
#include "groupnorm_two.h"
#include "launch.h"
#include "launchers.h"

namespace shai {

namespace {

// Registers allow 16 vectors of 4 channels a thread; with a fold's loads in flight beside them 8.  Two groups a workgroup leave half
// as many workgroups, and with 16 vectors it was the slower way (4 x 32 x 32 x 960: 14.8 us, statistics and apply 12.8; 4 x 48 x 48 x
// 320: 12.1 and 11.6; with 8, 4 x 16 x 16 x 960: 7.3 and 9.8).
constexpr int kMaxVec = 16, kMaxVecTwo = 8, kMaxVecFold = 8;
// Pixels of all parts, times a group's width and 160, from which the fold and the norm are two launches, the fold on every CU, where the
// one launch has up to 64 workgroups. What a pixel costs the one launch grows little with the width: it is a row of its own in every part.
// us with the convolution, one launch and two, above: 2 x 32 x 32 x 640 in 4 parts 54.3 and 48.2, 1 x 32 x 32 x 640 in 8 58.4 and 39.7, 2 x
// 24 x 24 x 640 in 4 42.8 and 41.6, 2 x 40 x 40 x 320 in 3 44.8 and 29.9, 1 x 16 x 16 x 1280 in 8 35.2 and 34.3, 2 x 16 x 16 x 1280 in 8
// 52.8 and 53.2, in 12 50.9 and 49.0, 2 x 20 x 20 x 1280 in 6 60.4 and 59.5; below: 2 x 16 x 16 x 640 in 8 26.9 and 27.0, 2 x 24 x 24 x 640
// in 3 47.7 and 47.5, 2 x 20 x 20 x 1280 in 4 69.5 and 70.3, 2 x 16 x 16 x 1280 in 6 38.2 and 39.8, 1 x 12 x 12 x 2560 in 8 34.6 and 38.5.
// With 96 and 128 workgroups: 3 x 16 x 16 x 1280 in 8 56.3 and 62.2, 4 x 16 x 16 x 1280 in 8 73.5 and 76.0, 4 x 24 x 24 x 640 in 6 58.0 and
// 58.3.
constexpr long kFoldTwo = 2048 * 200;
constexpr int kFoldTwoUnits = 64;

struct GnOneGeom {
  int u;        // groups per workgroup
  int vp;       // 4-channel vectors per pixel
  int nv;       // vectors per thread: 1, 2, 4, 8 or 16
  int active;   // threads with vectors, a multiple of vp: a thread's vectors are of the same channels
};

bool geometry(int HW, int C, int G, int max_vec, GnOneGeom* q) {
  if (G <= 0 || C % G != 0) return false;
  const int cg = C / G;
  if (cg < 4 || cg % 2 != 0) return false;
  q->u = cg % 4 == 0 ? 1 : 2;
  if (G % q->u != 0) return false;
  q->vp = q->u * cg / 4;
  if (q->vp > 1024) return false;
  const long items = (long)HW * q->vp;
  if (q->u == 2 && max_vec > kMaxVecTwo) max_vec = kMaxVecTwo;
  for (q->nv = 1; q->nv <= max_vec; q->nv *= 2) {
    const long need = (items + q->nv - 1) / q->nv;
    const long active = (need + q->vp - 1) / q->vp * q->vp;
    if (active <= 1024) {
      q->active = (int)active;
      return true;
    }
  }
  return false;
}

// Sums of lo and hi over the workgroup, the same value in every thread.
template <bool TWO>
__device__ __forceinline__ void block_sums(float& lo, float& hi, float2* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo += __shfl_xor(lo, o, 64);
    if constexpr (TWO) hi += __shfl_xor(hi, o, 64);
  }
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();                     // the last call's reads
  if ((threadIdx.x & 63) == 0) red[w] = make_float2(lo, hi);
  __syncthreads();
  lo = hi = 0.f;
  for (int i = 0; i < nw; ++i) {
    const float2 v = red[i];
    lo += v.x;
    if constexpr (TWO) hi += v.y;
  }
}

// PART: the workgroup has `len` pixels of its image, the unit's blockIdx-th of gridDim / (N units); it writes the fold to a.raw and its
// (mean, sum of squares about it) to stats [N, G, segments], and the rest is gn_apply_stats_kernel's.
template <int NV, bool TWO, bool FOLD, bool PART = false>
__global__ void __launch_bounds__(1024) gn_one_kernel(const GnOneArgs a, int units, int vp, int active, int len, float2* __restrict__ stats) {
  __shared__ float2 red[16];
  // neighbouring channels share cache lines: consecutive units of an image on one XCD
  int bid = blockIdx.x;
  if ((gridDim.x & 7) == 0) bid = (bid & 7) * (gridDim.x >> 3) + (bid >> 3);
  const int segs = PART ? (a.HW + len - 1) / len : 1;
  const int n = bid / (units * segs), seg = PART ? bid % segs : 0, unit = (bid - n * units * segs) / segs;
  const int t = threadIdx.x, cg = a.C / a.G;
  const bool live = t < active;
  const int end = PART ? min(a.HW, (seg + 1) * len) : a.HW;
  const int pix0 = t / vp + seg * len, cv = t % vp, step = active / vp;
  const int c = unit * vp * 4 + cv * 4;                       // first of the thread's 4 channels
  const int first = TWO ? min(4, max(0, cg - cv * 4)) : 4;    // how many of them are in the workgroup's first group

  uint2_ gm{}, bt{};
  if (live) {
    if (a.gamma) gm = *reinterpret_cast<const uint2_*>(a.gamma + c);
    if (a.beta) bt = *reinterpret_cast<const uint2_*>(a.beta + c);
  }
  uint2_ v[NV];
  if constexpr (!FOLD) {
    const bool one = c < a.C1;
    const int ld = one ? a.C1 : a.C - a.C1;
    const bf16_t* src = (one ? a.x + c : a.x2 + (c - a.C1)) + (long)n * a.HW * ld;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int p = pix0 + j * step;
      v[j] = live && p < end ? *reinterpret_cast<const uint2_*>(src + (long)p * ld) : uint2_{0, 0};
    }
  } else {
    // the split-K fold: parts in order, then bias, the image's bias, residual, as gemm_splitk_reduce does it
    constexpr int U = PART && NV == 1 ? 8 : NV <= 2 ? 4 : NV <= 4 ? 2 : 1;   // parts whose loads are in flight together
    const long slab = (long)a.N * a.HW * a.C;
    const float* src = a.parts + (long)n * a.HW * a.C + c;
    uint2_ rs[NV], bi{}, b2{};
    if (live) {
      if (a.bias) bi = *reinterpret_cast<const uint2_*>(a.bias + c);
      if (a.bias2d) b2 = *reinterpret_cast<const uint2_*>(a.bias2d + (long)n * a.bias2d_ld + c);
    }
    float4_ acc[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      acc[j] = float4_{0.f, 0.f, 0.f, 0.f};
      const int p = pix0 + j * step;
      rs[j] = a.residual && live && p < end ? *reinterpret_cast<const uint2_*>(a.residual + ((long)n * a.HW + p) * a.C + c) : uint2_{0, 0};
    }
    for (int s0 = 0; s0 < a.splits; s0 += U) {
      float4_ x[U][NV];
#pragma unroll
      for (int q = 0; q < U; ++q)
#pragma unroll
        for (int j = 0; j < NV; ++j) {
          const int p = pix0 + j * step;
          x[q][j] = live && p < end && s0 + q < a.splits ? *reinterpret_cast<const float4_*>(src + (s0 + q) * slab + (long)p * a.C)
                                                          : float4_{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
      for (int q = 0; q < U; ++q)
#pragma unroll
        for (int j = 0; j < NV; ++j) acc[j] += x[q][j];
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int p = pix0 + j * step;
      const bool in = live && p < end;
      float f[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int sh = e & 1 ? 0 : 16;
        auto part = [&](const uint2_& w) { return __uint_as_float(sh ? w[e >> 1] << 16 : w[e >> 1] & 0xffff0000u); };
        f[e] = acc[j][e];
        if (a.bias) f[e] += part(bi);
        if (a.bias2d) f[e] += part(b2);
        if (a.residual) f[e] += part(rs[j]) * a.res_alpha;
        if (!in) f[e] = 0.f;
      }
      v[j] = uint2_{pack2(f[0], f[1]), pack2(f[2], f[3])};
      if (a.raw && in) *reinterpret_cast<uint2_*>(a.raw + ((long)n * a.HW + p) * a.C + c) = v[j];
    }
  }

  auto at = [&](const uint2_& w, int e) { return __uint_as_float(e & 1 ? w[e >> 1] & 0xffff0000u : w[e >> 1] << 16); };
  const float inv = 1.f / ((float)(PART ? end - seg * len : a.HW) * (float)cg);
  float lo = 0.f, hi = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float f = at(v[j], e);
      if (!TWO || e < first) lo += f;
      else hi += f;
    }
  block_sums<TWO>(lo, hi, red);
  const float mlo = lo * inv, mhi = hi * inv;
  lo = hi = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if (!live || pix0 + j * step >= end) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool l = !TWO || e < first;
      const float d = at(v[j], e) - (l ? mlo : mhi);
      if (l) lo = fmaf(d, d, lo);
      else hi = fmaf(d, d, hi);
    }
  }
  block_sums<TWO>(lo, hi, red);
  if constexpr (PART) {
    if (t == 0) {
      float2* at = stats + ((long)n * a.G + unit * (TWO ? 2 : 1)) * segs + seg;
      at[0] = make_float2(mlo, lo);
      if constexpr (TWO) at[segs] = make_float2(mhi, hi);
    }
    return;
  }
  if (!live) return;
  const float rlo = rsqrtf(lo * inv + a.eps), rhi = rsqrtf(hi * inv + a.eps);
  float sc[4], sf[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const bool l = !TWO || e < first;
    sc[e] = (l ? rlo : rhi) * (a.gamma ? at(gm, e) : 1.f);
    sf[e] = (a.beta ? at(bt, e) : 0.f) - (l ? mlo : mhi) * sc[e];
  }
  bf16_t* dst = a.out + (long)n * a.HW * a.C + c;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int p = pix0 + j * step;
    if (p >= a.HW) continue;
    float y[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      y[e] = fmaf(at(v[j], e), sc[e], sf[e]);
      if (a.silu) y[e] = silu_f(y[e]);
    }
    *reinterpret_cast<uint2_*>(dst + (long)p * a.C) = uint2_{pack2(y[0], y[1]), pack2(y[2], y[3])};
  }
}

// y = (silu)((x - mean) rstd gamma + beta) from the segments' (mean, sum of squares about it), combined as Chan et al. do.  A workgroup
// makes its image's scale and shift of every channel in LDS, its pixels already on their way.
constexpr int kApplyC = 2560;                                // most channels
template <int V>                                             // vectors of 8 channels a thread has in flight
__global__ void __launch_bounds__(256) gn_apply_stats_kernel(const GnOneArgs a, const bf16_t* __restrict__ x, const float2* __restrict__ stats,
                                                             int segs, int len, int rows) {
  __shared__ float2 group[128];
  __shared__ float2 ss[kApplyC];
  const int C8 = a.C >> 3, cg = a.C / a.G, blocks = (a.HW + rows - 1) / rows;
  const int n = blockIdx.x / blocks, r0 = (blockIdx.x - n * blocks) * rows, r1 = min(a.HW, r0 + rows);
  const long base = ((long)n * a.HW + r0) * C8;
  const int total = (r1 - r0) * C8;
  const uint4_* src = reinterpret_cast<const uint4_*>(x) + base;
  uint4_* dst = reinterpret_cast<uint4_*>(a.out) + base;
  uint4_ v[V];
#pragma unroll
  for (int j = 0; j < V; ++j) {
    const int i = threadIdx.x + 256 * j;
    v[j] = src[min(i, total - 1)];
  }
  if ((int)threadIdx.x < a.G) {
    const float2* at = stats + ((long)n * a.G + threadIdx.x) * segs;
    float mean = 0.f, m2 = 0.f;
    for (int k = 0; k < segs; ++k) mean += at[k].x * (float)(min(a.HW, (k + 1) * len) - k * len);
    mean /= (float)a.HW;
    for (int k = 0; k < segs; ++k) {
      const float d = at[k].x - mean;
      m2 += at[k].y + d * d * (float)(min(a.HW, (k + 1) * len) - k * len) * (float)cg;
    }
    group[threadIdx.x] = make_float2(mean, rsqrtf(m2 / ((float)a.HW * (float)cg) + a.eps));
  }
  __syncthreads();
  for (int c = threadIdx.x; c < a.C; c += 256) {
    const float2 g = group[c / cg];
    const float sc = g.y * (a.gamma ? bf2f(a.gamma[c]) : 1.f);
    ss[c] = make_float2(sc, (a.beta ? bf2f(a.beta[c]) : 0.f) - g.x * sc);
  }
  __syncthreads();
  for (int i0 = 0; i0 < total; i0 += 256 * V) {
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const int i = i0 + threadIdx.x + 256 * j;
      if (i >= total) break;
      if (i0 > 0) v[j] = src[i];
      const int c = i % C8 * 8;
      float f[8];
      unpack8(v[j], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        f[e] = fmaf(f[e], ss[c + e].x, ss[c + e].y);
        if (a.silu) f[e] = silu_f(f[e]);
      }
      dst[i] = pack8(f);
    }
  }
}

// The fold's pixels are cut so that about every CU has a workgroup; a thread then has one vector of 4 channels, or two, of each part.
struct GnTwoGeom {
  GnOneGeom one;
  int len, segs;
};

bool two_geometry(const GnOneArgs& a, GnTwoGeom* q) {
  GnOneGeom whole;
  if (a.G > 128 || a.C > kApplyC || a.C % 8 != 0 || !geometry(a.HW, a.C, a.G, kMaxVec, &whole)) return false;
  const int units = a.N * (a.G / whole.u);
  int segs = (256 + units - 1) / units;
  if (segs > 16) segs = 16;
  q->len = (a.HW + segs - 1) / segs;
  q->segs = (a.HW + q->len - 1) / q->len;
  return q->segs > 1 && geometry(q->len, a.C, a.G, 2, &q->one);
}

}  // namespace

bool gn_one_supported(int HW, int C, int G, bool fold) {
  GnOneGeom q;
  return HW > 0 && geometry(HW, C, G, fold ? kMaxVecFold : kMaxVec, &q);
}

hipError_t launch_gn_one(const GnOneArgs& a, hipStream_t s) {
  GnOneGeom q;
  const bool fold = a.parts != nullptr;
  if (a.N <= 0) return hipSuccess;
  if (a.HW <= 0 || !geometry(a.HW, a.C, a.G, fold ? kMaxVecFold : kMaxVec, &q)) return hipErrorInvalidValue;
  const int units = a.G / q.u, threads = (q.active + 63) / 64 * 64;
  auto go = [&](auto kernel) { return launch(kernel, a.N * units, threads, s, a, units, q.vp, q.active, a.HW, (float2*)nullptr); };
#define SHAI_GN1(NV)                                                                                     \
  case NV:                                                                                               \
    return q.u == 2 ? go(fold ? gn_one_kernel<NV, true, true> : gn_one_kernel<NV, true, false>)          \
                    : go(fold ? gn_one_kernel<NV, false, true> : gn_one_kernel<NV, false, false>);
  switch (q.nv) {
    SHAI_GN1(1)
    SHAI_GN1(2)
    SHAI_GN1(4)
    SHAI_GN1(8)
    default:  // 16, of one group, never behind a fold
      return go(gn_one_kernel<16, false, false>);
  }
#undef SHAI_GN1
}

bool gn_two_wanted(const GnOneArgs& a) {
  GnTwoGeom q;
  return a.parts != nullptr && (long)a.HW * a.splits * (a.C / a.G + 160) >= kFoldTwo && ((uintptr_t)a.out & 15) == 0 && two_geometry(a, &q) &&
         a.N * (a.G / q.one.u) <= kFoldTwoUnits;
}

long gn_two_floats(const GnOneArgs& a) {
  GnTwoGeom q;
  return two_geometry(a, &q) ? 2L * a.N * a.G * q.segs : 0;
}

hipError_t launch_gn_two(const GnOneArgs& a, bf16_t* raw, float* stats, hipStream_t s) {
  GnTwoGeom q;
  if (a.parts == nullptr || !two_geometry(a, &q)) return hipErrorInvalidValue;
  if (a.N <= 0) return hipSuccess;
  GnOneArgs f = a;
  f.raw = raw;
  const int units = a.G / q.one.u, threads = (q.one.active + 63) / 64 * 64;
  auto go = [&](auto kernel) {
    return launch(kernel, a.N * units * q.segs, threads, s, f, units, q.one.vp, q.one.active, q.len, (float2*)stats);
  };
  const hipError_t e = q.one.u == 2 ? (q.one.nv == 1 ? go(gn_one_kernel<1, true, true, true>) : go(gn_one_kernel<2, true, true, true>))
                                    : (q.one.nv == 1 ? go(gn_one_kernel<1, false, true, true>) : go(gn_one_kernel<2, false, true, true>));
  if (e != hipSuccess) return e;
  const int rows = (int)((long)a.N * a.HW + 255) / 256;      // of an image a workgroup
  const int blocks = (a.HW + rows - 1) / rows;
  return launch(gn_apply_stats_kernel<4>, a.N * blocks, 256, s, a, (const bf16_t*)raw, (const float2*)stats, q.segs, q.len, rows);
}

}  // namespace shai
