// One step's attention of a kv head over a paged cache (attn.hip says how), for the kernels that hold it.
#pragma once
#include "lm_device.h"
#include "lm.h"

namespace shai_lm {

constexpr float kLog2e = 1.4426950408889634f;

// the first key that position pos sees
__device__ __forceinline__ int first_key(const AttnArgs& p, int pos) {
  return p.window ? max(0, pos - p.chunk + 1) : pos - pos % p.chunk;
}

// 8 consecutive elements
__device__ __forceinline__ void load8(const bf16_t* p, float* x) { unpack8(*reinterpret_cast<const uint4_*>(p), x); }
__device__ __forceinline__ void load8(const float* p, float* x) {
  *reinterpret_cast<float4_*>(x) = load4(p);
  *reinterpret_cast<float4_*>(x + 4) = load4(p + 4);
}
__device__ __forceinline__ void store8(bf16_t* p, const float* x) { *reinterpret_cast<uint4_*>(p) = pack8(x); }
__device__ __forceinline__ void store8(float* p, const float* x) {
  store4(p, *reinterpret_cast<const float4_*>(x));
  store4(p + 4, *reinterpret_cast<const float4_*>(x + 4));
}

// One head by n / 8 lanes of a wave, lane j holding elements 8 j .. 8 j + 7: dimension i < rot / 2 turned with i + rot / 2 by
// the row's angles, then the head divided by its root mean square over `dim` (the pads behind are zero); with `gain` the norm
// comes first.  `stage`: n floats of LDS.  Every lane of the wave calls it.
__device__ __forceinline__ void turn_and_norm(float (&x)[8], float* stage, const float* rope, int rot, int dim, float eps,
                                              int j, int lanes, const float* gain) {
  const int half = rot >> 1;
  if (gain) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += x[i] * x[i];
    for (int o = lanes >> 1; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
    const float r = 1.f / sqrtf(ss / (float)dim + eps);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] *= r * gain[8 * j + i];
  }
  store8(stage + 8 * j, x);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int e = 8 * j + i;
    if (e < rot) {
      const bool low = e < half;
      const float other = stage[low ? e + half : e - half];
      const float* t = rope + 2 * (low ? e : e - half);
      x[i] = x[i] * t[0] + (low ? -other : other) * t[1];
    }
    ss += x[i] * x[i];
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (gain) return;
  for (int o = lanes >> 1; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
  const float r = 1.f / sqrtf(ss / (float)dim + eps);
#pragma unroll
  for (int i = 0; i < 8; ++i) x[i] *= r;
}

// what a head's summed output is multiplied by: the denominator L (of exponents to the base 2 above M) with its sink, the gate
__device__ __forceinline__ float out_factor(const AttnArgs& p, const bf16_t* row, int h, int d, float M, float L) {
  float up = p.gate_w ? sigmoid_f(bf2f(row[p.gate_off + (long)h * p.gate_w + (p.gate_w > 1 ? d : 0)])) : p.out_scale;
  if (p.sink) {
    const float sk = p.sink[h] * kLog2e, top = fmaxf(M, sk), a = __builtin_amdgcn_exp2f(M - top);
    L = L * a + __builtin_amdgcn_exp2f(sk - top);
    up *= a;
  }
  return up / L;
}

// One workgroup: kv head g's query heads h0 .. h0 + R - 1 (R <= 16, RH = R rounded up) of sequence b, one split of the
// visible 64-key blocks.  Wave w takes blocks w, w + 4, ... of the split.  VMAX: most V loads in flight.
template <int DK, int DV, int RH, bool PREP, int VMAX>
__device__ __forceinline__ void attn_decode(const AttnArgs& p, int per_group, int store, int bx, int b, int split) {
  constexpr int LPK = DV / 8, KP = 64 / LPK, IT = 64 / KP;   // V: LPK lanes per key, KP keys at a time
  constexpr int VB = IT > VMAX ? VMAX : IT;                  // V loads in flight
  __shared__ float sp[4][64][RH];
  __shared__ __attribute__((aligned(16))) float so[4][RH][DV];
  __shared__ __attribute__((aligned(16))) bf16_t sq[PREP ? RH : 1][PREP ? DK : 8];
  static_assert(!PREP || 4 * RH * DV >= (RH + 1) * DK, "prepared heads are staged in so");
  __shared__ float sm[4][16], sl[4][16];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int c = lane & 15, q4 = lane >> 4;
  const int group = p.H / p.G, parts = (group + per_group - 1) / per_group;
  const int g = bx / parts, part = bx % parts;
  const int h0 = g * group + part * per_group, R = min(per_group, group - part * per_group);
  const int pos = p.ctx[b] - 1, lo = first_key(p, pos);
  const int b0 = lo >> 6, b1 = (pos >> 6) + 1;
  const int per = (b1 - b0 + p.splits - 1) / p.splits;
  const int s0 = b0 + split * per, s1 = min(b1, s0 + per);
  const bf16_t* row = static_cast<const bf16_t*>(p.qkvg) + (long)b * p.ld;
  bf16_t* kc = static_cast<bf16_t*>(p.kc);
  bf16_t* vc = static_cast<bf16_t*>(p.vc);

  // this step's k / v: stored by the only workgroup that reads them (the one with the last block)
  const int slot = p.slots[b];
  if (store && slot >= 0 && s1 == b1 && s0 < s1) {
    const long cell = ((long)(slot >> 6) * p.G + g) * 64 + (slot & 63);
    const bf16_t* kn = row + (long)p.H * DK + (long)g * DK;
    const bf16_t* vn = row + p.v_off + (long)g * DV;
    if (tid < DK / 8) {
      if constexpr (!PREP) reinterpret_cast<uint4_*>(kc + cell * DK)[tid] = reinterpret_cast<const uint4_*>(kn)[tid];
    } else if (tid >= 64 && tid - 64 < DV / 8)
      reinterpret_cast<uint4_*>(vc + cell * DV)[tid - 64] = reinterpret_cast<const uint4_*>(vn)[tid - 64];
  }
  if constexpr (PREP) {                          // the heads of this workgroup, and k where it is stored
    constexpr int LPH = DK / 8, HP = 256 / LPH;
    const bool key = store && slot >= 0 && s1 == b1 && s0 < s1;
    const int n = R + key, j = tid % LPH;
    for (int i0 = 0; i0 < n; i0 += HP) {
      const int i = i0 + tid / LPH, ii = min(i, n - 1);
      float x[8];
      load8(row + (long)(ii < R ? h0 + ii : p.H + g) * DK + 8 * j, x);
      // the spare lanes repeat the last head with the same values
      turn_and_norm(x, &so[0][0][0] + ii * DK, p.rope + (long)b * p.rot, p.rot, p.dim, p.eps, j, LPH,
                    ii < R ? p.q_gain : p.k_gain);
      if (i < R) store8(&sq[i][8 * j], x);
      else if (i < n) store8(kc + (((long)(slot >> 6) * p.G + g) * 64 + (slot & 63)) * DK + 8 * j, x);
    }
  }
  __syncthreads();

  uint4_ qf[DK / 64][2];
#pragma unroll
  for (int s = 0; s < DK / 64; ++s)
#pragma unroll
    for (int u = 0; u < 2; ++u)
      qf[s][u] = c < R ? *reinterpret_cast<const uint4_*>((PREP ? &sq[min(c, RH - 1)][0] : row + (long)(h0 + c) * DK) +
                                                          64 * s + 16 * q4 + 8 * u)
                       : uint4_{0u, 0u, 0u, 0u};
  float o[RH][8];
#pragma unroll
  for (int r = 0; r < RH; ++r)
#pragma unroll
    for (int j = 0; j < 8; ++j) o[r][j] = 0.f;
  float m = -INFINITY, l = 0.f;                  // of head c (replicated over q4)
  const float sl2 = p.scale * kLog2e * (p.temp ? p.temp[h0 + min(c, R - 1)] : 1.f);
  const int vk = lane / LPK, vcol = (lane % LPK) * 8;

  for (int kb = s0 + w; kb < s1; kb += 4) {
    const long cell = ((long)p.bt[(long)b * p.max_blocks + kb] * p.G + g) * 64;
    const bf16_t* kp = kc + (cell + c) * DK + 16 * q4;
    const bf16_t* vp = vc + (cell + vk) * DV + vcol;
    float4_ s[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      s[t] = float4_{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < DK / 64; ++d)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const uint4_ kf = *reinterpret_cast<const uint4_*>(kp + (long)16 * t * DK + 64 * d + 8 * u);
          s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, kf),
                                                         __builtin_bit_cast(bf16x8, qf[d][u]), s[t], 0, 0, 0);
        }
    }
    uint4_ v[VB];
#pragma unroll
    for (int i = 0; i < VB; ++i) v[i] = *reinterpret_cast<const uint4_*>(vp + (long)i * KP * DV);
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kb * 64 + 16 * t + 4 * q4 + i;
        s[t][i] = key < lo || key > pos ? -INFINITY : s[t][i] * sl2;
        mx = fmaxf(mx, s[t][i]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float mn = fmaxf(m, mx);               // finite: every visited block holds a visible key
    const float alpha = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(s[t][i] - mn);
        sum += e;
        if (c < RH) sp[w][16 * t + 4 * q4 + i][c] = e;
      }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    l = l * alpha + sum;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int r = 0; r < RH; ++r) {
      const float ar = __shfl(alpha, r, 64);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[r][j] *= ar;
    }
#pragma unroll
    for (int i0 = 0; i0 < IT; i0 += VB) {
      if (i0 > 0) {
#pragma unroll
        for (int i = 0; i < VB; ++i) v[i] = *reinterpret_cast<const uint4_*>(vp + (long)(i0 + i) * KP * DV);
      }
#pragma unroll
      for (int i = 0; i < VB; ++i) {
        float f[8];
        unpack8(v[i], f);
        const float* pr = &sp[w][(i0 + i) * KP + vk][0];
#pragma unroll
        for (int r = 0; r < RH; ++r) {
          const float pv = pr[r];
#pragma unroll
          for (int j = 0; j < 8; ++j) o[r][j] = fmaf(pv, f[j], o[r][j]);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
  // fold the key lanes of the wave, then the waves
#pragma unroll
  for (int r = 0; r < RH; ++r)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float x = o[r][j];
#pragma unroll
      for (int d = LPK; d < 64; d <<= 1) x += __shfl_xor(x, d, 64);
      if (vk == 0) so[w][r][vcol + j] = x;
    }
  if (lane < 16) {
    sm[w][lane] = m;
    sl[w][lane] = l;
  }
  __syncthreads();
  for (int i = tid; i < R * DV; i += 256) {
    const int r = i / DV, d = i - r * DV, h = h0 + r;
    const float M = fmaxf(fmaxf(sm[0][r], sm[1][r]), fmaxf(sm[2][r], sm[3][r]));
    float L = 0.f, x = 0.f;
    if (M > -INFINITY) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float e = __builtin_amdgcn_exp2f(sm[k][r] - M);
        L += sl[k][r] * e;
        x += so[k][r][d] * e;
      }
    }
    if (p.splits == 1) {
      static_cast<bf16_t*>(p.o)[(long)b * p.ldo + h * DV + d] = f2bf(x * out_factor(p, row, h, d, M, L));
    } else {
      float* ws = p.ws + (((long)b * p.H + h) * p.splits + split) * (DV + 2);
      ws[d] = x;
      if (d == 0) {
        ws[DV] = M;
        ws[DV + 1] = L;
      }
    }
  }
}

}  // namespace shai_lm
