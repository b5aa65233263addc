// C = epi(A W^T) for few rows of A (decode steps of a batch: up to 64) with bf16 weights; gemm_ring_fits says from how many on.
//
// The streaming kernel (gemm.hip) reads both operands straight into registers, 16 rows x 16 bytes per quarter wave: 14 bytes per
// clock and CU, of which A, the same for every workgroup, is as much as W at 64 rows.  DMA to LDS moves 30.  So here both
// operands go through a ring in LDS, 128 k at a time, and one workgroup per CU owns as many columns as give every CU one
// (16 NT; A is read once per CU): 17424 x 2048 on 64 rows is 228 workgroups of 80 columns (5 blocks of 16), 32768 x 2048 is 256 of 128.
//
// 8 waves: wave w takes the 32 k of sub-step w % 4 and the row blocks of half w / 4; the four k-groups' sums meet in LDS and are
// added in their order.  Rows past M or N and values past K are out of the buffers' range: zeros, no traffic.
// Where a row of W is a multiple of 4 KB, a workgroup with all of K begins kTurn steps behind the one before it and goes round: begun together,
// all of them read the same columns of W from a part of the memory's channels.  us in order -> turned, cold weights, 16 / 32 / 64 rows: 8192 x 8192
// 34.6 / 40.0 / 38.9 -> 26.8 / 26.6 / 33.3, 17424 x 2048 19.1 / 19.6 / 21.9 -> 16.7 / 17.2 / 20.4, 32768 x 2048 35.1 / 33.5 / 37.3 -> 35.4 / 33.5 / 29.6,
// 28672 x 4096 53.9 / 57.0 / 54.0 -> 50.6 / 50.8 / 53.0, 8192 x 14336 (112 steps, 16 beginnings) 48.4 / 51.6 / 63.5 -> 44.2 / 48.3 / 62.0, 8192 x 6144 23.2 /
// 24.7 / 30.5 -> 20.9 / 22.7 / 29.5; 8192 x 8192 on 16 rows by one step 35.2, by three 29.9, by five 27.1.  Other rows gain nothing by it and took longer: 5632 x
// 1024 5.8 / 6.1 / 6.9 -> 6.0 / 6.4 / 7.2, 9216 x 3072 13.9 / 15.8 / 20.5 -> 14.4 / 16.1 / 20.8, 8192 x 3584 13.4 / 14.6 / 18.9 -> 14.0 / 14.9 / 19.1.
//
// LDS rows are 256 bytes; chunk c (16 bytes) of row r is at c ^ (r & 15): no bank conflicts, and the DMA stays lane-linear because
// the source address carries the permutation.
//
// Replays of a HIP graph over weights larger than the caches, us (streaming kernel -> here; N x K, 64 rows): 17424 x 2048
// 26.2 -> 20.5, 32768 x 2048 42.3 -> 29.7, 24576 x 4096 69.3 -> 42.1, 8256 x 2048 18.0 -> 14.5, 4096 x 2048 11.0 -> 10.0, partial
// sums of 2048 x 12544 21.6 (4 parts) -> 14.5 (8 parts).  17424 x 2048 is 71 MB: 3.5 TB/s.  What is left is the start (launch, the
// first stage's latency) and the joining of the sums, about 5 us, and the memory's rate in between.
#include "lm_device.h"
#include "lm.h"

#include <type_traits>

namespace shai_lm {

namespace {

constexpr uint32_t kOob = 0x80000000u;
constexpr int KS = 128;                       // k of one ring stage
constexpr unsigned kTurn = 7;                 // steps by which a workgroup begins behind the one before it

constexpr int ring_stages(int MT, int NT) {   // as many as fit in 160 KB, at most 5
  const int n = 160 * 1024 / ((MT + NT) * 16 * KS * 2);
  return n < 5 ? n : 5;
}

template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <typename O, int EC, int MT, int NT>
__global__ void __launch_bounds__(512) gemm_ring_kernel(const GemmArgs p) {
  constexpr int S = ring_stages(MT, NT), STAGE = (MT + NT) * 16 * KS;  // elements
  constexpr int PIECES = 4 * (MT + NT);       // DMA instructions of a stage (4 rows each): W's, then A's
  constexpr int HI = (PIECES + 7) / 8, LO = PIECES / 8, MH = MT / 2;
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4, kg = wid & 3, mh = wid >> 2;
  const int n0 = blockIdx.x * 16 * NT;
  const __amdgpu_buffer_rsrc_t rw = rsrc(p.W, (long)p.N * p.K * 2), ra = rsrc(p.A, ((long)(p.M - 1) * p.lda + p.K) * 2);
  int first = 0, steps = (p.K + KS - 1) / KS;
  O* C = static_cast<O*>(p.C);
  if (p.splits > 1) {
    const int all = steps;
    first = (int)(blockIdx.y * (long)all / p.splits);
    steps = (int)((blockIdx.y + 1L) * all / p.splits) - first;
    C += (long)blockIdx.y * p.M * p.N;
  }
  const int turn = p.splits > 1 || p.K % 2048 != 0 ? 0 : (int)(blockIdx.x * kTurn % steps);   // the first step
  uint32_t off[HI];
  int col[HI];                                // first k of this lane's chunk within a stage
#pragma unroll
  for (int j = 0; j < HI; ++j) {
    const int piece = wid + 8 * j, row = (piece < 4 * NT ? piece : piece - 4 * NT) * 4 + g;
    col[j] = (r ^ (row & 15)) * 8;
    if (piece < 4 * NT) off[j] = n0 + row < p.N ? (uint32_t)(((long)(n0 + row) * p.K + col[j]) * 2) : kOob;
    else off[j] = row < p.M ? (uint32_t)(((long)row * p.lda + col[j]) * 2) : kOob;
  }
  auto stage = [&](int buf, int s) {          // step s of this workgroup; past its end: zeros
    const int k = (first + (s + turn < steps ? s + turn : s + turn - steps)) * KS;
#pragma unroll
    for (int j = 0; j < HI; ++j) {
      const int piece = wid + 8 * j;
      if (j < LO || piece < PIECES) {
        const uint32_t o = s < steps && k + col[j] < p.K ? off[j] + (uint32_t)(k * 2) : kOob;
        dma16(piece < 4 * NT ? rw : ra, lds + buf * STAGE + piece * 512, o);
      }
    }
  };
  float4_ acc[NT][MH];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MH; ++j) acc[i][j] = float4_{0.f, 0.f, 0.f, 0.f};
  auto frag = [&](const bf16_t* base, int block) {
    return *reinterpret_cast<const bf16x8*>(base + (block * 16 + r) * KS + (((kg * 4 + g) ^ r) * 8));
  };
#pragma unroll
  for (int s = 0; s < S - 1; ++s) stage(s, s);
  int buf = 0;
  for (int s = 0; s < steps; ++s) {
    if (wid < PIECES % 8) wait_vm<(S - 2) * HI>();
    else wait_vm<(S - 2) * LO>();
    __builtin_amdgcn_s_barrier();             // every wave's part of the step is there, and the buffer before it has been read
    stage(buf == 0 ? S - 1 : buf - 1, s + S - 1);
    const bf16_t *w = lds + buf * STAGE, *a = w + NT * 16 * KS;
    bf16x8 fw[NT], fa[MH];
#pragma unroll
    for (int j = 0; j < MH; ++j) fa[j] = frag(a, mh * MH + j);
#pragma unroll
    for (int i = 0; i < NT; ++i) fw[i] = frag(w, i);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MH; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[i], fa[j], acc[i][j], 0, 0, 0);
    buf = buf == S - 1 ? 0 : buf + 1;
  }
  wait_vm<0>();
  __syncthreads();
  static_assert(4 * NT * MT * 1024 <= S * STAGE * 2, "partial sums larger than the ring");
  float4_* red = reinterpret_cast<float4_*>(lds);  // [k-group][block][lane]
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MH; ++j) red[((kg * NT + i) * MT + mh * MH + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  for (int t = wid; t < NT * MT; t += 8) {
    float4_ c = red[t * 64 + lane];
#pragma unroll
    for (int q = 1; q < 4; ++q) c += red[(q * NT * MT + t) * 64 + lane];
    const int m = t % MT * 16 + r;
    if (m < p.M) store_cols<O, EC>(p, C, m, n0 + t / MT * 16 + 4 * g, c);
  }
}

template <typename O, int EC, int MT>
void launch_blocks(const GemmArgs& a, int nt, hipStream_t s) {
  auto go = [&](auto kernel, int NT) {
    const size_t bytes = (size_t)ring_stages(MT, NT) * (MT + NT) * 16 * KS * 2;
    kernel<<<dim3((a.N + 16 * NT - 1) / (16 * NT), a.splits > 1 ? a.splits : 1), 512, bytes, s>>>(a);
  };
  switch (nt) {
    case 2: go(gemm_ring_kernel<O, EC, MT, 2>, 2); break;
    case 3: go(gemm_ring_kernel<O, EC, MT, 3>, 3); break;
    case 4: go(gemm_ring_kernel<O, EC, MT, 4>, 4); break;
    case 5: go(gemm_ring_kernel<O, EC, MT, 5>, 5); break;
    case 6: go(gemm_ring_kernel<O, EC, MT, 6>, 6); break;
    default: go(gemm_ring_kernel<O, EC, MT, 8>, 8); break;
  }
  SHAI_CHECK_LAUNCH();
}

}  // namespace

// Columns of a workgroup, in blocks of 16: one workgroup per CU, or as few rounds of them as 128 columns allow.  Up to 32 rows a
// stage is short, and beyond one round of 112 columns two workgroups of 48 per CU, each other's prologue and end hidden, are
// faster (50176 x 4096, 32 rows: 88.9 us; one of 128: 91.8).  That was so of all before workgroups began at different steps of K; since
// then 32768 x 2048 is 33.1 us in 48 columns and 28.2 in 128, x 3072 45.7 and 40.2, x 4096 56.3 and 56.0.
constexpr long kRound = 256 * 112;
static int ring_blocks(const GemmArgs& a) {
  const long cols = (long)a.N * (a.splits > 1 ? a.splits : 1), rounds = (cols + 256 * 128 - 1) / (256 * 128);
  if (a.M <= 32 && cols > kRound) return 3;
  const int nt = (int)((cols + 256 * 16 * rounds - 1) / (256 * 16 * rounds));
  return nt < 2 ? 2 : nt > 6 ? 8 : nt;
}

// Where the ring was no slower than the streaming kernel, whose 16-column workgroups read few rows of A from few cache lines, start
// faster, and have no sums to join.  Replays of a HIP graph, cold weights, N x K (streaming -> ring, us):
//   from 4097 columns on, which are more 16-column workgroups than CUs: 9 rows, from 7169 on 12.  These lines were drawn when all workgroups
//     began at column 0 (8192 x 8192: 9 rows 1.05 of the time, 12 1.04, 16 0.94).  Now the ring is ahead on both sides of them: 5120 x 2048, 1 row
//     0.87, 9 0.80; 8192 x 8192, 1 0.91, 9 0.83, 12 0.77, 16 0.70; 17424 x 2048, 1 0.96, 9 0.86, 16 0.74; 9216 x 3072, 1 0.82, 12 0.71; 14336 x 5120, 1 0.93,
//     12 0.70; 28672 x 4096 alone 1 1.29, 9 1.08, 12 0.99.  Up to eleven rows they stand where they were: in whole steps only 1 row was
//     timed with the ring, where most of such products are normed_gemm's, without a gain;
//   below: 33 rows from 2049 columns on (2304 x 4096, 64 rows: 23.9 -> 15.3; 2048 x 2048 8.4 -> 9.4), and 17 to 32 rows where M K >=
//     24 * 1024 (2048 x 2048, 32 rows: 8.3 -> 7.6; 4096 x 1024: 17 rows 1.04 of the time, 24 rows 1.00);
//   partial sums: more than 16 rows (512 x 8448 in 8 parts, 17 rows: 6.8 -> 5.8); up to 16 of a K of 4096, from 2049 columns on, or
//     where 32-column workgroups of all parts fill 7 of 8 CUs and either 9 rows or a K of 8192 are there: 2048 x 8448 in 4 parts,
//     1 row 10.2 -> 9.4, 16 rows 11.4 -> 9.3; x 6144, 9 rows 8.1 -> 7.5; 1024 x 12544 in 8, 1 row 8.0 ->
//     7.9, 16 rows 9.1 -> 7.8; with half of the CUs the streaming kernel's 16 columns are faster: 512 x 8448 in 8, 1 row 4.8 -> 5.3.
//   Up to 32 rows more columns than one round of 112 (ring_blocks) take a K, or part of one, of 3072: 32768 x 1024, 32 rows 1.14 of
//     the time, x 2048 0.99, x 4096 0.89; 8192 x 2048 in 4 parts, 8 rows 15.6 -> 19.0.
// Products per head, grouped by expert or longer than a buffer's range stay with the streaming kernel.
bool gemm_ring_fits(const GemmArgs& a) {
  const long lim = 0x7fffffffL, splits = a.splits > 1 ? a.splits : 1;
  if (a.tiles || a.batch > 1 || a.M > 64 || a.K < 512 || a.N < 512 || (long)a.N * a.K * 2 >= lim || (long)a.M * a.lda * 2 >= lim)
    return false;
  if (a.M <= 32 && a.N * splits > kRound && a.K / splits < 3072) return false;
  if (splits > 1) return a.M > 16 || (a.K >= 4096 && (a.N > 2048 || (a.N * splits >= 224 * 32 && (a.M > 8 || a.K >= 8192))));
  if (a.N > 4096) return a.M >= (a.N <= 7168 ? 9 : 12);
  return a.M > 32 ? a.N > 2048 : a.M > 16 && a.M * a.K >= 24 * 1024;
}

void launch_gemm_ring(const GemmArgs& a, hipStream_t s) {
  const int nt = ring_blocks(a), ec = epi_class(a.epi);
  auto rows = [&](auto o, auto c) {
    using O = decltype(o);
    if (a.M <= 32) launch_blocks<O, decltype(c)::value, 2>(a, nt, s);
    else launch_blocks<O, decltype(c)::value, 4>(a, nt, s);
  };
#define CLASS(EC_) std::integral_constant<int, EC_>()
  if (a.out_f32 && ec == EC_PLAIN) rows(float(), CLASS(EC_PLAIN));
  else if (a.out_f32) rows(float(), CLASS(EC_ANY));
  else if (ec == EC_PLAIN) rows(bf16_t(), CLASS(EC_PLAIN));
  else if (ec == EC_CLAMP) rows(bf16_t(), CLASS(EC_CLAMP));
  else if (ec == EC_GELU) rows(bf16_t(), CLASS(EC_GELU));
  else rows(bf16_t(), CLASS(EC_OTHER));
#undef CLASS
}

}  // namespace shai_lm
