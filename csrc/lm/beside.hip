// A decode step of a layer's two mixers in one launch: attention over a paged cache (attn_decode.h) and the delta rule (rule_rows.h),
// which read different columns of the layer's rows and write different columns of its outputs.
//
// One after the other, an attention of a few workgroups waits for its chain of loads (block table, keys, values: 11.6 us for 132 keys and
// one sequence, 15.2 for 64 sequences, 0.25 to 1.3 TB/s), and then the recurrence begins.  Here the attention's workgroups are the first of
// the grid, so that their chains start at once, and the recurrence's, bound by the state's traffic, take the rest of the chip (kernels of
// one sequence 25.3 -> 16.5 us with what prepares them, of 64 sequences 1.0 of 33.9 ms a pass).
#include "attn_decode.h"
#include "rule_rows.h"

namespace shai_lm {

// Workgroups a CU that the registers are for: three, and two where eight heads of 128 to a group hold 198 of them.  The recurrence alone has
// 128, for four.  Given to both, with half as many V loads in flight, nothing spills either, but the attention's chain is the longer and
// decides (us, 16 heads of 128, 4 a group: one sequence of 132 keys 12.7 at three and 13.9 at four, 64 of 900 keys 59.1 and 68.1).  Eight a group at
// three spill 51 to 53: 64 sequences of 900 keys 72.9, at two 50.8, one after the other 67.4; of 132 keys 39.5, 36.7 and 45.7.
constexpr int workgroups(int D, int RH) { return D == 128 && RH == 8 ? 2 : 3; }

// V: V loads of the attention in flight. Eight where three workgroups share a CU: sixteen spill 7 registers there (64 sequences of 132 keys, 4 heads
// of 128 a group, 39.4 -> 38.3 us).
template <int D, int RH, int MODE, int SD, int V, int LOW = 0>
__global__ void __launch_bounds__(256, V == 16 ? 2 : workgroups(D, RH)) attn_rule_kernel(const AttnArgs a, const RuleArgs r, int per_group, int heads, int n_attn) {
  const int i = blockIdx.x;
  if (i < n_attn) {
    const int j = i / heads;
    attn_decode<D, D, RH, true, V>(a, per_group, 1, i - j * heads, j % a.B, j / a.B);
  } else {
    const int b = (i - n_attn) / r.H;
    rule_rows<bf16_t, MODE, SD, SD, 256, true, LOW>(r, i - n_attn - b * r.H, b);
  }
}

// Steps of up to so many workgroups have two on a CU at most, whatever their registers: sixteen loads without a spill (one sequence of 132 keys 12.9 ->
// 12.4 us).
constexpr int kFew = 512;

template <int D, int RH, int MODE, int SD>
static void attn_rule(const AttnArgs& a, const RuleArgs& r, hipStream_t s) {
  const int n_attn = a.G * a.B * a.splits, grid = n_attn + r.H * r.B;
  auto go = [&](auto kernel) { kernel<<<grid, 256, 0, s>>>(a, r, a.H / a.G, a.G, n_attn); };
  if constexpr (D == 128 && RH == 4) {
    if constexpr (MODE == kChannel && SD == 128) {
      if (r.up) return grid <= kFew ? go(attn_rule_kernel<D, RH, MODE, SD, 16, 1>) : go(attn_rule_kernel<D, RH, MODE, SD, 8, 2>);
    }
    if (grid <= kFew) return go(attn_rule_kernel<D, RH, MODE, SD, 16>);
  }
  go(attn_rule_kernel<D, RH, MODE, SD, 8>);
}

template <int D, int RH>
static void attn_rule(const AttnArgs& a, const RuleArgs& r, hipStream_t s) {
  if (r.mode == kHead) r.dk == 64 ? attn_rule<D, RH, kHead, 64>(a, r, s) : attn_rule<D, RH, kHead, 128>(a, r, s);
  else r.dk == 64 ? attn_rule<D, RH, kChannel, 64>(a, r, s) : attn_rule<D, RH, kChannel, 128>(a, r, s);
}

// The head sizes and groups that are compiled; others run one after the other.
static bool fits(const AttnArgs& a, const RuleArgs& r) {
  const long grid = (long)a.G * a.B * a.splits + (long)r.H * r.B;
  return a.own_kv && a.rope && a.H / a.G <= 8 && a.dk == a.dv && a.dk <= 128 && r.mode != kRetention && r.dk == r.dv && r.dk <= 128 &&
         r.q_lens == nullptr && grid <= 0x7fffffffL;
}

// The logits of gates and decays in this launch: an attention of few sequences takes longer than the recurrence beside it, so that their product (64 KB
// of weights a head from the XCD's cache) costs little there and a launch of its own less; where three workgroups share a CU they hide it from each
// other, with the state asked for behind the weights, in the registers that these had.  us apart and in one, 16 heads, ranks of 128: one sequence of 132
// keys 15.3 and 11.5, 8 16.4 and 13.1, 25 26.3 and 22.0; 32 30.5 and 28.3, 64 46.2 and 42.8, 96 (1920 workgroups) 60.2 and 59.8; of 900 keys 64 69.1 and
// 67.4; of one key 64 30.6 and 30.9, 96 41.3 and 43.9: up to two rounds of three to a CU.
constexpr int kLow = 2 * 3 * 256;
bool attn_rule_low_fits(const AttnArgs& a, const RuleArgs& r, bool f32) {
  const auto rank = [](int n) { return n == 64 || n == 128; };
  return !f32 && fits(a, r) && a.dk == 128 && a.H / a.G <= 4 && r.mode == kChannel && r.dk == 128 && rank(r.low_a) && rank(r.low_g) &&
         r.ldg % 8 == 0 && (((uintptr_t)r.gate | (uintptr_t)r.up) & 15) == 0 && (long)a.G * a.B * a.splits + (long)r.H * r.B <= kLow;
}

void launch_attn_beside_rule(const AttnArgs& a, const RuleArgs& r, bool f32, hipStream_t s) {
  if (f32 || !fits(a, r)) {
    launch_attn_decode(a, f32, s);
    launch_rule_rows(r, f32, s);
    return;
  }
  const bool few = a.H / a.G <= 4;
  if (a.dk == 64) few ? attn_rule<64, 4>(a, r, s) : attn_rule<64, 8>(a, r, s);
  else few ? attn_rule<128, 4>(a, r, s) : attn_rule<128, 8>(a, r, s);
  if (a.splits > 1) launch_attn_decode_fold(a, s);
  SHAI_CHECK_LAUNCH();
}

}  // namespace shai_lm
