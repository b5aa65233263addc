// The four-wave tile (gemm_w4_kernel.h): 256 x 256 products and convolutions.
#include "gemm_w4_kernel.h"

namespace shai {

bool gemm_w4_supported(const GemmArgs& a) {
  if (a.in_scale != nullptr || a.rms || a.w_scale != nullptr || (a.glu && a.N % 8 != 0)) return false;
  if (a.K % 8 != 0 || a.lda % 8 != 0 || a.ldw % 8 != 0) return false;  // 16-B source chunks
  if ((long)a.N * a.ldw * 2 >= 0x7fffffffL) return false;
  if (a.conv) {
    if (a.Cin % 64 != 0 || (a.A2 != nullptr && a.Cin1 % 64 != 0)) return false;
    if (a.act != ACT_NONE && a.act != ACT_SILU) return false;  // the conv branch instantiates these two only
    return (long)a.Nimg * a.H * a.Wd * a.Cin * 2 < 0x7fffffffL;
  }
  return a.A2 == nullptr && (long)a.M * a.lda * 2 < 0x7fffffffL;
}

// bn: columns of a tile, 256 or 192 (products only)
void launch_gemm_w4(const GemmArgs& a, int bn, hipStream_t s) {
  if (!a.conv) {
    if (bn == 192) launch_gemm_w4_narrow(a, s);
    else w4_product<8, 8>(a, s);
    return;
  }
  if (a.upsample) {
    if (a.act == ACT_SILU) w4_go<8, 8, 2, false, ACT_SILU>(a, s);
    else w4_go<8, 8, 2, false, ACT_NONE>(a, s);
  } else {
    if (a.act == ACT_SILU) w4_go<8, 8, 1, false, ACT_SILU>(a, s);
    else w4_go<8, 8, 1, false, ACT_NONE>(a, s);
  }
}

}  // namespace shai
