// lanes.h -- exchanges of doubles between the lanes of a wave by VALU moves
// (DPP and the half and row swaps of gfx950), without the LDS round trip of
// ds_bpermute that __shfl takes (device code).
#pragma once

#include <hip/hip_runtime.h>

namespace yh {

// v of the lane that DPP control CTRL names, 0 where it names none: 0x100 + n
// the lane n up in its row of 16.
template <int CTRL>
__device__ __forceinline__ double dpp_double(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Swaps the upper half of a with the lower half of b, or (ROWS) rows 1 and 3
// of a with rows 0 and 2 of b.
template <bool ROWS>
__device__ __forceinline__ void swap_lanes(double& a, double& b) {
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  const auto lo = ROWS ? __builtin_amdgcn_permlane16_swap((int)x, (int)y, false, false)
                       : __builtin_amdgcn_permlane32_swap((int)x, (int)y, false, false);
  const auto hi = ROWS ? __builtin_amdgcn_permlane16_swap((int)(x >> 32), (int)(y >> 32), false, false)
                       : __builtin_amdgcn_permlane32_swap((int)(x >> 32), (int)(y >> 32), false, false);
  a = __longlong_as_double(((long long)hi[0] << 32) | (unsigned)lo[0]);
  b = __longlong_as_double(((long long)hi[1] << 32) | (unsigned)lo[1]);
}

// Sum over a row of 16 lanes in its first lane: v0 + v8, then + v4 + v12, ...
__device__ __forceinline__ double row_sum(double v) {
  v += dpp_double<0x108>(v);
  v += dpp_double<0x104>(v);
  v += dpp_double<0x102>(v);
  v += dpp_double<0x101>(v);
  return v;
}

// Sum over the wave in lane 0, with the pairs of a __shfl_down tree (32, 16,
// ... 1), so with its bits.
__device__ __forceinline__ double wave_sum(double v) {
  double a = v, b = v;
  swap_lanes<false>(a, b);
  v = a + b;  // lane i < 32: v[i] + v[i + 32]
  a = b = v;
  swap_lanes<true>(a, b);
  return row_sum(a + b);
}

}  // namespace yh
