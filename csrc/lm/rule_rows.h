// The recurrences of rule.hip row by row: a workgroup has a head of a sequence, for the kernels that hold it.
#pragma once
#include "matrix_state.h"
#include "lm.h"

namespace shai_lm {

constexpr int kRetention = 0, kHead = 1, kChannel = 2;     // decay: fixed; per head; per key channel
constexpr float kLeast = -40.f;                            // base-2 logarithm of a decay that leaves nothing in fp32

__device__ __forceinline__ float softplus_exact(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }
template <bool FAST>
__device__ __forceinline__ float gate_act(float z, int kind) {
  const float s = FAST ? __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-z * kInvLn2)) : sigmoid_f(z);
  return kind == 0 ? z * s : s;
}

// ------------------------------------------------------------------------------------------------ row by row
// Thread: 4 columns x DK / RG rows of S.  S^T k and S^T q are taken from the decayed state in one pass: with kq = k . q,
// o = S^T q + kq u.
//
// Decode: every workgroup of a step is resident at once, so whatever stands between the state's arrival and its way back is time
// in which memory idles.  A wave's loads return in order; everything small is therefore loaded first, without branches (the
// convolution's taps one after the other, each waited for, cost 10 us of a step), and the state after it: convolutions, norms and
// decays are done when it arrives.  64 sequences x 16 heads of 128 x 128 (134 MB of state),
// us: decay per head 37.6 -> 34.8, per channel 39.8 -> 35.1, retention 28.7 (the rate of a large copy: 27); one sequence 7.1 -> 6.6 and
// 7.6 -> 6.8.  The one row of a step is compiled apart from prompts': 126 registers instead of 168, four workgroups per CU
// (three beside a step's attention, beside.hip: 64 sequences are then more than are resident at once).
// LOW: gate and decay logits are products of the row's low_a + low_g values with this head's rows of `up`, 16 rows a matrix instruction, the
// same values in all its columns (as bf16 for the gate, as the product apart leaves them).  1: the state is on its way meanwhile, 2: asked for
// behind them, in the registers they had.
template <typename T, int MODE, int DK, int DV, int NT, bool STEP, int LOW = 0>   // STEP: decode of the delta rule
__device__ __forceinline__ void rule_rows(const RuleArgs& p, int h, int b) {
  constexpr bool DELTA = MODE != kRetention;
  constexpr int NC = DV / 4, RG = NT / NC, R = DK / RG, NW = NT / 64, KW = DK / 64;
  static_assert(R % 4 == 0 && NC <= 64 && NT >= DV && NT >= 2 * DK, "shape");
  __shared__ __attribute__((aligned(16))) float sq[DK], sk[DK], sg[MODE == kChannel ? DK : 4], sv[DV];
  __shared__ __attribute__((aligned(16))) float sa[DELTA ? NW : 1][DV], so[NW][DV];
  __shared__ float red[NW], skq[NW], rout[NW];
  static_assert(!LOW || (STEP && MODE == kChannel && DK == 128 && DV == 128 && NT == 256), "two waves for decays and two for gates");
  __shared__ __attribute__((aligned(16))) float slow[LOW ? DK + DV : 4];   // this head's decay logits, then its gates
  const int tid = threadIdx.x;
  const int c = (tid % NC) * 4, r0 = (tid / NC) * R;
  const int n = !STEP && p.q_lens ? p.q_lens[b] : 1;
  if (n < 1) return;
  const long t0 = !STEP && p.q_start ? p.q_start[b] : b;
  const int slot = p.slots[b], pos0 = p.pos[t0];
  const int g = h / (p.H / p.G), channels = 2 * p.G * DK + p.H * DV;
  float* st = p.state + (((long)max(slot, 0) * p.H + h) * DK + r0) * DV + c;
  const bool old = slot >= 0 && pos0 > 0;
  const T* x = static_cast<const T*>(p.x);
  T* ring = DELTA ? static_cast<T*>(p.ring) + (long)max(slot, 0) * p.taps * channels : nullptr;
  const int ring0 = DELTA ? pos0 % p.taps : 0;
  // The newest inputs of a channel and their taps; the others are added by `conv`.  A step's loads are issued whatever the taps: only
  // taps that there are count for a prompt, whose rows come one after the other (fp32, 2 x 200 rows, 16 heads of 128 x 128, 1 tap: 697
  // -> 574 us, 4 taps 696 -> 698).
  constexpr int NEAR = 4;
  struct Near {
    T x[NEAR];
    float w[NEAR];
  };
  auto source = [&](long t, int ch, int j, bool& valid) {    // input j rows before row t
    const int row = STEP ? 0 : (int)(t - t0), m = ring0 + row - j;      // before the step's first row: its place in the ring
    const bool here = row >= j;
    valid = j < p.taps && (here || (pos0 + row >= j && slot >= 0));
    return here || !valid ? x + (valid ? t - j : t) * p.ldx + ch : ring + (m < 0 ? m + p.taps : m) * channels + ch;
  };
  auto near = [&](long t, int ch) {
    Near a{};
#pragma unroll
    for (int j = 0; j < NEAR; ++j) {
      bool valid;
      if (!STEP && j >= p.taps) break;
      a.x[j] = *source(t, ch, j, valid);
      a.w[j] = p.conv[max(p.taps - 1 - j, 0) * channels + ch];
    }
    return a;
  };
  // channel ch of row t after its convolution and silu
  auto conv = [&](long t, int ch, const Near& a) {
    float y = a.w[0] * load1(&a.x[0]);
#pragma unroll
    for (int j = 1; j < NEAR; ++j) {
      bool valid;
      if (!STEP && j >= p.taps) break;
      source(t, ch, j, valid);
      if (valid) y += a.w[j] * load1(&a.x[j]);
    }
    for (int j = NEAR; j < p.taps; ++j) {
      bool valid;
      const T* src = source(t, ch, j, valid);
      if (valid) y += p.conv[(p.taps - 1 - j) * channels + ch] * load1(src);
    }
    return silu_exact(y);
  };
  const bool key = tid >= DK;
  const int my_d = key ? tid - DK : tid, my_ch = (key ? p.G + g : g) * DK + my_d;   // delta rule: this thread's q or k channel
  const int v_ch = 2 * p.G * DK + h * DV + tid;
  struct Small {             // what a row needs besides the state
    Near qk, v;
    float decay, bias, beta;
    T gate;
  };
  auto small = [&](long t) {
    Small s{};
    if constexpr (DELTA) {
      if (tid < 2 * DK) s.qk = near(t, my_ch);
      if (tid < DV) s.v = near(t, v_ch);
      s.beta = p.beta[t * p.ldb + h];
      const int d = MODE == kChannel ? h * DK + min(tid, DK - 1) : h;
      if constexpr (!LOW) s.decay = p.decay[t * p.ldd + d];
      s.bias = p.bias[d];
    }
    if (!LOW && tid < DV) s.gate = static_cast<const T*>(p.gate)[t * p.ldg + h * DV + tid];
    return s;
  };
  Small in{};
  if constexpr (STEP) in = small(t0);
  const float rate = p.rate[h];
  __builtin_amdgcn_sched_barrier(0);
  [[maybe_unused]] uint4_ lw[LOW ? 4 : 1][4], lx[4];            // 4 blocks of 16 rows of `up`, 32 of up to 128 columns each
  if constexpr (LOW) {
    const int w = tid >> 6, r = tid & 15, q = tid >> 4 & 3;
    const bool decays = w < 2;
    const int rank = decays ? p.low_a : p.low_g, col = (decays ? 0 : p.low_a) + 8 * q;
    const long row = (decays ? (long)p.H * DV + h * DK + w * 64 : (long)h * DV + (w - 2) * 64) + r;
    const bf16_t* up = static_cast<const bf16_t*>(p.up) + row * (p.low_a + p.low_g) + col;
    const bf16_t* low = static_cast<const bf16_t*>(p.gate) + t0 * p.ldg + col;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = min(32 * s, rank - 32);
      lx[s] = *reinterpret_cast<const uint4_*>(low + k);
      if (32 * s >= rank) lx[s] = uint4_{0u, 0u, 0u, 0u};
#pragma unroll
      for (int i = 0; i < 4; ++i) lw[i][s] = *reinterpret_cast<const uint4_*>(up + (long)(16 * i) * (p.low_a + p.low_g) + k);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  float4_ S[R];
  auto ask = [&] {
#pragma unroll
    for (int i = 0; i < R; ++i) S[i] = old ? load4(st + (long)i * DV) : float4_{0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (LOW != 2) ask();
  if constexpr (LOW) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float4_ y = float4_{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) y = mac(__builtin_bit_cast(bf16x8, lw[i][s]), __builtin_bit_cast(bf16x8, lx[s]), y);
      if ((tid & 15) == 0) store4(slow + (tid >> 6) * 64 + 16 * i + 4 * (tid >> 4 & 3), y);
    }
    if constexpr (LOW == 2) {
      __builtin_amdgcn_sched_barrier(0);
      ask();
    }
    __syncthreads();
  }
  for (long t = t0; t < t0 + n; ++t) {
    const T* row = x + t * p.ldx;
    if constexpr (!STEP) in = small(t);
    float mine = 0.f;
    if (tid < 2 * DK) {
      const int d = my_d, first = DELTA ? my_ch - my_d : (key ? p.H + h : h) * DK;
      if constexpr (DELTA) {
        mine = conv(t, my_ch, in.qk);
      } else {
        mine = load1(row + first + d);
        if (d < p.rot) {
          const int half = p.rot >> 1;
          const bool low = d < half;
          const float other = load1(row + first + (low ? d + half : d - half));
          const float* a = p.rope + t * p.rot + 2 * (low ? d : d - half);
          mine = mine * a[0] + (low ? -other : other) * a[1];
        }
      }
      (key ? sk : sq)[d] = mine;
    }
    if constexpr (DELTA) {
      const float ss = wave_sum(mine * mine);
      if ((tid & 63) == 0) red[tid >> 6] = ss;
    }
    const int v0 = (DELTA ? 2 * p.G * DK : 2 * p.H * DK) + h * DV;
    if (tid < DV) sv[tid] = DELTA ? conv(t, v_ch, in.v) : load1(row + v0 + tid);
    if constexpr (MODE == kChannel) {
      if (tid < DK) sg[tid] = expf(-rate * softplus_exact((LOW ? slow[tid] : in.decay) + in.bias));
    }
    __syncthreads();
    float rq = 1.f, rk = 1.f, gh = MODE == kRetention ? rate : 1.f, beta = 1.f;
    if constexpr (DELTA) {
      float s0 = 0.f, s1 = 0.f;
#pragma unroll
      for (int w = 0; w < KW; ++w) {
        s0 += red[w];
        s1 += red[KW + w];
      }
      rq = 1.f / sqrtf(s0 + 1e-6f) * (1.f / sqrtf((float)p.dim));
      rk = 1.f / sqrtf(s1 + 1e-6f);
      beta = sigmoid_f(in.beta);
      if constexpr (MODE == kHead) gh = expf(-rate * softplus_exact(in.decay + in.bias));
    } else {
      rk = 1.f / sqrtf((float)p.dim);
    }
    const float4_ v = load4(sv + c);
    float4_ a = float4_{0.f, 0.f, 0.f, 0.f}, o = a;
    float kq = 0.f;
#pragma unroll
    for (int i = 0; i < R; i += 4) {
      __builtin_amdgcn_sched_barrier(0);          // four rows of k and q in registers at a time
      const float4_ k = load4(sk + r0 + i) * rk, q = load4(sq + r0 + i) * rq;
      const float4_ f = MODE == kChannel ? load4(sg + r0 + i) : float4_{gh, gh, gh, gh};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        S[i + j] = f[j] * S[i + j];
        if constexpr (DELTA) {
          a += k[j] * S[i + j];
          kq += k[j] * q[j];
        } else {
          S[i + j] += k[j] * v;
        }
        o += q[j] * S[i + j];
      }
    }
#pragma unroll
    for (int d = NC; d < 64; d <<= 1) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (DELTA) a[j] += __shfl_xor(a[j], d, 64);
        o[j] += __shfl_xor(o[j], d, 64);
      }
      if constexpr (DELTA) kq += __shfl_xor(kq, d, 64);
    }
    if ((tid & 63) < NC) {
      if constexpr (DELTA) store4(&sa[tid >> 6][c], a);
      store4(&so[tid >> 6][c], o);
    }
    if (DELTA && (tid & 63) == 0) skq[tid >> 6] = kq;
    __syncthreads();
    float y = 0.f;
    if (tid < DV) {
#pragma unroll
      for (int w = 0; w < NW; ++w) y += so[w][tid];
    }
    if constexpr (DELTA) {
      float4_ sum = float4_{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w) sum += load4(&sa[w][c]);
      const float4_ u = beta * (v - sum);
#pragma unroll
      for (int i = 0; i < R; i += 4) {
        __builtin_amdgcn_sched_barrier(0);
        const float4_ k = load4(sk + r0 + i) * rk;
#pragma unroll
        for (int j = 0; j < 4; ++j) S[i + j] += k[j] * u;
      }
      if (tid < DV) {
        float all = 0.f, s = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          all += skq[w];
          s += sa[w][tid];
        }
        y += all * beta * (sv[tid] - s);
      }
    }
    const float ss = wave_sum(y * y);
    if ((tid & 63) == 0) rout[tid >> 6] = ss;
    __syncthreads();
    if (tid < DV) {
      float sum = 0.f;
#pragma unroll
      for (int w = 0; w < DV / 64; ++w) sum += rout[w];
      const float z = LOW ? bf2f(f2bf(slow[DK + tid])) : load1(&in.gate);
      const float r = 1.f / sqrtf(sum / (float)p.vdim + p.eps);
      store1(static_cast<T*>(p.out) + t * p.ldo + h * DV + tid, y * r * (DELTA ? p.gain[tid] : 1.f) * gate_act<false>(z, p.gate_kind));
    }
  }
  if (slot >= 0) {
#pragma unroll
    for (int i = 0; i < R; ++i) store4(st + (long)i * DV, S[i]);
    if (DELTA && !p.q_lens) {                     // this step's inputs, where no workgroup of the step reads
      T* to = ring + (long)(pos0 % p.taps) * channels;
      const T* row = x + t0 * p.ldx;
      if (tid < 2 * DK && h % (p.H / p.G) == 0) {
        const int ch = (tid >= DK ? p.G + g : g) * DK + (tid >= DK ? tid - DK : tid);
        to[ch] = row[ch];
      }
      const int ch = 2 * p.G * DK + h * DV + tid;
      if (tid < DV) to[ch] = row[ch];
    }
  }
}

}  // namespace shai_lm
