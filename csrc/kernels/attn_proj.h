// Attention of short sequences with its output projection (attn_proj.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace shai {
typedef uint16_t bf16_t;

// parts[h] = softmax(scale q_h k_h^T (+ bias_h)) v_h W_h^T, W_h the 64 columns of W that head h's output meets
struct AttnProjArgs {
  const bf16_t* q;       // [B, Sq, H, 64], k / v [B, Skv, H, 64]: heads packed, rows and batches apart by these strides
  const bf16_t* k;
  const bf16_t* v;
  long q_bs, q_ts, k_bs, k_ts, v_bs, v_ts;
  const int* kv_lens;    // [B] or null
  const bf16_t* bias;    // [H, Sq, Skv] or null
  const bf16_t* W;       // [N, H * 64], rows ldw apart
  long ldw;
  float* parts;          // [H, B * Sq, N]
  int B, H, Sq, Skv, N, causal;
  float scale;
};
// up to 256 keys, N a multiple of 16, every address and stride of 16 bytes
bool attn_proj_supported(const AttnProjArgs& a);
[[nodiscard]] hipError_t launch_attn_proj(const AttnProjArgs& a, hipStream_t s);
}  // namespace shai
