// A wave's search over a launch's table (device code).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tsa {
namespace dev {

// The last of n entries (ascending first(i), n > 0) whose first is at most s; 0 if none is. The wave's 64 lanes probe
// together, so 64 entries cost one memory latency; all of them call it with the same arguments.
template <class F>
__device__ __forceinline__ uint32_t last_at_most(uint32_t n, uint64_t s, F first) {
  uint32_t lo = 0, hi = n;
  while (hi - lo > 1) {
    const uint32_t step = (hi - lo + 63) / 64, at = lo + (threadIdx.x & 63u) * step;
    const bool under = at >= lo && at < hi && first(at) <= s;
    const uint32_t k = uint32_t(__popcll(__ballot(under)));
    lo += (k ? k - 1 : 0) * step;
    hi = hi - lo < step ? hi : lo + step;
  }
  return lo;
}

}  // namespace dev
}  // namespace tsa
