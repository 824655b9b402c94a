// Device helpers shared by the selector's files: walking the elements of 64
// sets at a time, block maxima of argmax keys.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device_util.h"

namespace rip {

// Each lane of a wave holds one run (off, len) of `data`; the wave visits
// every element of the 64 runs once, lanes taking elements of any run:
// f(value, run index).
template <typename F>
__device__ inline void for_each_run_element(unsigned long long off, uint32_t len,
                                            const uint32_t *data, uint32_t *s_pre,
                                            unsigned long long *s_off, F &&f) {
  const uint32_t lane = lane_id();
  s_off[lane] = off;
  const uint32_t incl = wave_inclusive_scan(len);
  s_pre[lane + 1] = incl;
  if (lane == 0) s_pre[0] = 0;
  const uint32_t total = __shfl(incl, 63, 64);
  __builtin_amdgcn_wave_barrier();
  for (uint32_t i = lane; i < total; i += 64) {
    uint32_t lo = 0, hi = 64;
    while (lo < hi) {
      const uint32_t mid = (lo + hi) >> 1;
      if (s_pre[mid + 1] <= i) lo = mid + 1;
      else hi = mid;
    }
    f(data[s_off[lo] + (i - s_pre[lo])], lo);
  }
  __builtin_amdgcn_wave_barrier();
}

__device__ inline unsigned long long wave_max_u64(unsigned long long x) {
  for (int d = 32; d > 0; d >>= 1) {
    const unsigned long long y = __shfl_xor(x, d, 64);
    x = y > x ? y : x;
  }
  return x;
}

// Blocks of a grid over `work` items, per_block each, at most cap (at least 1).
inline uint32_t grid_for(uint64_t work, uint32_t per_block, uint32_t cap) {
  const uint64_t g = (work + per_block - 1) / per_block;
  return static_cast<uint32_t>(std::max<uint64_t>(1, std::min<uint64_t>(g, cap)));
}

}  // namespace rip
