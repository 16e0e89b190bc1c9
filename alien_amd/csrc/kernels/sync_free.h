// Bit patterns of the sync-free sweeps: a value is ready when it is not the sentinel.
#pragma once

#include <hip/hip_runtime.h>

namespace alien_hip {

template <typename T> struct SfBits;
template <> struct SfBits<double> {
  typedef unsigned long long U;
  static constexpr U kSentinel = 0x7ff4deadbeef0001ull; // a signalling NaN: never an arithmetic result
  static __device__ __forceinline__ U bits(double v) { return (U)__double_as_longlong(v); }
  static __device__ __forceinline__ double value(U b) { return __longlong_as_double((long long)b); }
};
template <> struct SfBits<float> {
  typedef unsigned int U;
  static constexpr U kSentinel = 0x7fa5deadu;
  static __device__ __forceinline__ U bits(float v) { return __float_as_uint(v); }
  static __device__ __forceinline__ float value(U b) { return __uint_as_float(b); }
};

} // namespace alien_hip
