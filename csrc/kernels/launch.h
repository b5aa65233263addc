// A kernel launch with its own status, for launchers whose caller reports it.
#pragma once
#include <hip/hip_runtime.h>

namespace shai {

template <class... P>
[[nodiscard]] inline hipError_t launch(void (*kernel)(P...), unsigned grid, unsigned block, hipStream_t s, P... a) {
  void* args[] = {&a...};
  return hipLaunchKernel(reinterpret_cast<const void*>(kernel), dim3(grid), dim3(block), args, 0, s);
}

}  // namespace shai
