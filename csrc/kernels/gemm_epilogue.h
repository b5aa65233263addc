// Shared GEMM epilogue (v2 LDS-DMA GEMM, pipelined 256x256 GEMM, split-K fold).
#pragma once
#include "common.h"
#include "launchers.h"

namespace shai {

// Phase-decomposed upsample conv (GemmArgs::upsample == 2, gemm_8ph.hip CONV 3), row order: groups of
// G = max(1, 256 / (H W)) images (H, W powers of two, host-checked); inside a group phase-major (ph = 2 py + px), then
// image, then (i, j) of the low-resolution grid.  A 256-row tile so holds ONE phase (its weight slice); G = 1 is
// image-major.  Shifts only: the epilogue evaluates this per stored row.
struct Up2Row {
  int img, ph, si, sj;
};
__device__ __forceinline__ Up2Row up2_row(const GemmArgs& p, int m) {
  const int lw = __builtin_ctz((unsigned)p.Wd), lhw = lw + __builtin_ctz((unsigned)p.H);
  const int lb = lhw >= 8 ? lhw : 8;  // log2 of one (group, phase) block's rows, G H W
  const int r = m & ((1 << lb) - 1), r2 = r & ((1 << lhw) - 1);
  Up2Row q;
  q.ph = (m >> lb) & 3;
  q.img = ((m >> (lb + 2)) << (lb - lhw)) + (r >> lhw);
  q.si = r2 >> lw;
  q.sj = r2 & (p.Wd - 1);
  return q;
}
// the output pixel row of GEMM row m (epilogue and split-K fold)
__device__ __forceinline__ long up2_out_row(const GemmArgs& p, int m) {
  const Up2Row q = up2_row(p, m);
  return ((long)q.img * p.OH + 2 * q.si + (q.ph >> 1)) * p.OW + 2 * q.sj + (q.ph & 1);
}

// Apply the epilogue to 4 consecutive columns n..n+3 of row m and store.
template <bool GLU, int ACT>
__device__ __forceinline__ void epilogue4(const GemmArgs& p, bf16_t* C, const bf16_t* R, int m, int n, float v[4],
                                          int b = 0) {
  const bool full = n + 3 < p.N && (p.ldc & 3) == 0 && (p.ldr & 3) == 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] *= p.alpha;
  if (p.bias) {
    if (full) {
      const uint2_ bb = *reinterpret_cast<const uint2_*>(p.bias + n);
      v[0] += bf2f(bb[0] & 0xffff); v[1] += bf2f(bb[0] >> 16);
      v[2] += bf2f(bb[1] & 0xffff); v[3] += bf2f(bb[1] >> 16);
    } else {
      for (int e = 0; e < 4 && n + e < p.N; ++e) v[e] += bf2f(p.bias[n + e]);
    }
  }
  if (p.bias2d) {
    const bf16_t* b2 = p.bias2d + (long)(m / p.rows_per_bias2d) * p.bias2d_ld;
    if (full && (p.bias2d_ld & 3) == 0) {
      const uint2_ bb = *reinterpret_cast<const uint2_*>(b2 + n);
      v[0] += bf2f(bb[0] & 0xffff); v[1] += bf2f(bb[0] >> 16);
      v[2] += bf2f(bb[1] & 0xffff); v[3] += bf2f(bb[1] >> 16);
    } else {
      for (int e = 0; e < 4 && n + e < p.N; ++e) v[e] += bf2f(b2[n + e]);
    }
  }
  const bf16_t* gr = p.gate ? p.gate + ((long)b * p.M + m) / p.rows_per_gate * p.gate_stride : nullptr;
  if constexpr (GLU) {
    float o0 = v[0] * apply_act<ACT>(v[1]);
    float o1 = v[2] * apply_act<ACT>(v[3]);
    const int nc = n >> 1;
    if (gr) {
      o0 *= bf2f(gr[nc]);
      o1 *= bf2f(gr[nc + 1]);
    }
    float r0 = 0.f, r1 = 0.f;
    if (R) {
      r0 = bf2f(R[(long)m * p.ldr + nc]) * p.res_alpha;
      r1 = bf2f(R[(long)m * p.ldr + nc + 1]) * p.res_alpha;
    }
    if (((p.ldc | nc) & 1) == 0) {
      *reinterpret_cast<uint32_t*>(C + (long)m * p.ldc + nc) = pack2(o0 + r0, o1 + r1);
    } else {
      C[(long)m * p.ldc + nc] = f2bf(o0 + r0);
      C[(long)m * p.ldc + nc + 1] = f2bf(o1 + r1);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = apply_act<ACT>(v[e]);
    if (gr) {
      for (int e = 0; e < 4 && n + e < p.N; ++e) v[e] *= bf2f(gr[n + e]);
    }
    if (full) {
      if (R) {
        const uint2_ rr = *reinterpret_cast<const uint2_*>(R + (long)m * p.ldr + n);
        v[0] += bf2f(rr[0] & 0xffff) * p.res_alpha; v[1] += bf2f(rr[0] >> 16) * p.res_alpha;
        v[2] += bf2f(rr[1] & 0xffff) * p.res_alpha; v[3] += bf2f(rr[1] >> 16) * p.res_alpha;
      }
      uint2_ o;
      o[0] = pack2(v[0], v[1]);
      o[1] = pack2(v[2], v[3]);
      *reinterpret_cast<uint2_*>(C + (long)m * p.ldc + n) = o;
    } else {
      for (int e = 0; e < 4 && n + e < p.N; ++e) {
        float x = v[e];
        if (R) x += bf2f(R[(long)m * p.ldr + n + e]) * p.res_alpha;
        C[(long)m * p.ldc + n + e] = f2bf(x);
      }
    }
  }
}

// Whether the width, and rows and bases of everything epilogue8 touches, allow its accesses: 16 bytes, or 8 for the output side of a GLU.
template <bool GLU>
inline bool epilogue8_fits(const GemmArgs& a) {
  constexpr int OUT = GLU ? 4 : 8;  // columns stored per call
  long rows = a.ldc;
  uintptr_t out = (uintptr_t)a.C;
  if (a.residual) rows |= a.ldr, out |= (uintptr_t)a.residual;
  if (a.gate) rows |= a.gate_stride, out |= (uintptr_t)a.gate;
  if (a.bias2d && (a.bias2d_ld & 7)) return false;
  if (a.batch > 1) rows |= a.batch_c | (a.residual ? a.batch_r : 0);
  return a.N % 8 == 0 && (rows & (OUT - 1)) == 0 && (out & (2 * OUT - 1)) == 0 && (((uintptr_t)a.bias | (uintptr_t)a.bias2d) & 15) == 0;
}

template <int V>
__device__ __forceinline__ void load_bf(const bf16_t* src, float (&x)[V]) {
  if constexpr (V == 8) {
    const uint4_ t = *reinterpret_cast<const uint4_*>(src);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = bf2f(e & 1 ? t[e >> 1] >> 16 : t[e >> 1] & 0xffff);
  } else {
    const uint2_ t = *reinterpret_cast<const uint2_*>(src);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = bf2f(e & 1 ? t[e >> 1] >> 16 : t[e >> 1] & 0xffff);
  }
}

// epilogue4 for the 8 consecutive columns n .. n + 7 of row m, all below N, with epilogue8_fits true: the same operations in
// the same order, one 16-byte access (8 bytes on the output side of a GLU) instead of two.
template <bool GLU, int ACT>
__device__ __forceinline__ void epilogue8(const GemmArgs& p, bf16_t* C, const bf16_t* R, int m, int n, float (&v)[8], int b) {
  float x[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] *= p.alpha;
  if (p.bias) {
    load_bf<8>(p.bias + n, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += x[e];
  }
  if (p.bias2d) {
    load_bf<8>(p.bias2d + (long)(m / p.rows_per_bias2d) * p.bias2d_ld + n, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += x[e];
  }
  constexpr int OUT = GLU ? 4 : 8;
  const int nc = GLU ? n >> 1 : n;
  float o[OUT], y[OUT];
#pragma unroll
  for (int e = 0; e < OUT; ++e) {
    if constexpr (GLU) o[e] = v[2 * e] * apply_act<ACT>(v[2 * e + 1]);
    else o[e] = apply_act<ACT>(v[e]);
  }
  if (p.gate) {
    load_bf<OUT>(p.gate + ((long)b * p.M + m) / p.rows_per_gate * p.gate_stride + nc, y);
#pragma unroll
    for (int e = 0; e < OUT; ++e) o[e] *= y[e];
  }
  if (R) {
    load_bf<OUT>(R + (long)m * p.ldr + nc, y);
#pragma unroll
    for (int e = 0; e < OUT; ++e) o[e] += y[e] * p.res_alpha;
  }
  if constexpr (GLU) {
    *reinterpret_cast<uint2_*>(C + (long)m * p.ldc + nc) = uint2_{pack2(o[0], o[1]), pack2(o[2], o[3])};
  } else {
    *reinterpret_cast<uint4_*>(C + (long)m * p.ldc + nc) =
        uint4_{pack2(o[0], o[1]), pack2(o[2], o[3]), pack2(o[4], o[5]), pack2(o[6], o[7])};
  }
}

}  // namespace shai
