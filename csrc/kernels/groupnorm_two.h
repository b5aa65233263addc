// GroupNorm behind the fold of a split convolution, in two launches (groupnorm.hip).
#pragma once
#include "launchers.h"

namespace shai {

// Whether the fold (GnOneArgs::parts) is large enough for it, and the floats of its workspace
bool gn_two_wanted(const GnOneArgs& a);
long gn_two_floats(const GnOneArgs& a);
// raw: [N, HW, C], receives the folded convolution
[[nodiscard]] hipError_t launch_gn_two(const GnOneArgs& a, bf16_t* raw, float* stats, hipStream_t s);

}  // namespace shai
