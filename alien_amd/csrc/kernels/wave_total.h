// Wavefront sums on every lane, bit for bit wave_sum's (device_common.h).
#pragma once

#include <hip/hip_runtime.h>

namespace alien_hip {

// Sum over the wavefront on every lane, by the tree of wave_sum (device_common.h: lanes 32, 16, .. 1
// apart): the lanes are paired both ways, inside the vector unit (about 30 cycles a step; __shfl
// goes through LDS, over 100).
struct Halves {
  unsigned lo, hi;
};
__device__ __forceinline__ Halves halves(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  return {(unsigned)b, (unsigned)(b >> 32)};
}
__device__ __forceinline__ double whole(unsigned lo, unsigned hi) {
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) {
  const Halves h = halves(v);
  return v + whole((unsigned)__builtin_amdgcn_update_dpp(0, (int)h.lo, CTRL, 0xf, 0xf, true),
                   (unsigned)__builtin_amdgcn_update_dpp(0, (int)h.hi, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ double wave_total(double v) {
  Halves h = halves(v);
  auto lo = __builtin_amdgcn_permlane32_swap(h.lo, h.lo, false, false); // lanes 0-31 twice, lanes 32-63 twice
  auto hi = __builtin_amdgcn_permlane32_swap(h.hi, h.hi, false, false);
  v = whole(lo[0], hi[0]) + whole(lo[1], hi[1]);
  h = halves(v);
  lo = __builtin_amdgcn_permlane16_swap(h.lo, h.lo, false, false); // even rows of 16 twice, odd rows twice
  hi = __builtin_amdgcn_permlane16_swap(h.hi, h.hi, false, false);
  v = whole(lo[0], hi[0]) + whole(lo[1], hi[1]);
  v = dpp_add<0x128>(v); // row rotated by 8
  v = dpp_add<0x124>(v); // by 4: lanes 8 apart hold the same by now
  v = dpp_add<0x4e>(v);  // quads 2 3 0 1
  return dpp_add<0xb1>(v); // 1 0 3 2
}

} // namespace alien_hip
