// The four-wave tile (gemm_w4_kernel.h): 256 x 192 products, a source of their own as they take minutes to compile.
#include "gemm_w4_kernel.h"

namespace shai {

void launch_gemm_w4_narrow(const GemmArgs& a, hipStream_t s) { w4_product<8, 6>(a, s); }

}  // namespace shai
