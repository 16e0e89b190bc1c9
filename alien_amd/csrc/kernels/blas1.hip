// BLAS-1 kernels of the HIP backend: the vector operations that
// CBLASMPIKernel (simple_csr/algebra/CBLASMPIKernel.h:37-125) and the SYCL
// KernelInternal (sycl/algebra/SYCLKernelInternal.h:110-246) provide.
//
// All element-wise operations round exactly like the sequential reference
// loops (built with -ffp-contract=off: no fused multiply-add). Each lane
// handles kEPT elements spaced one workgroup apart (coalesced), loading all of
// them before using any. Dot products accumulate in FP64 in one launch and
// leave the scalar in device memory (partials + launch_finalize).
#include "../alien_hip_internal.h"
#include "device_common.h"
#include "launch.h"
#include "wave_total.h"

namespace alien_hip {

#define EPT_INDEX(k) (blockIdx.x * (long)(kBlock * kEPT) + (k) * kBlock + threadIdx.x)

template <typename T>
__global__ void __launch_bounds__(kBlock) k_copy(int n, const T* __restrict__ x, T* __restrict__ y) {
#pragma unroll
  for (int k = 0; k < kEPT; ++k) {
    const long i = EPT_INDEX(k);
    if (i < n) y[i] = x[i];
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_axpy(int n, T a, const T* __restrict__ x, T* __restrict__ y) {
#pragma unroll
  for (int k = 0; k < kEPT; ++k) {
    const long i = EPT_INDEX(k);
    if (i < n) y[i] = y[i] + a * x[i];
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_scal(int n, T a, T* __restrict__ x) {
#pragma unroll
  for (int k = 0; k < kEPT; ++k) {
    const long i = EPT_INDEX(k);
    if (i < n) x[i] = a * x[i];
  }
}

template <typename T>
__global__ void __launch_bounds__(kBlock) k_assign(int n, T a, T* __restrict__ x) {
#pragma unroll
  for (int k = 0; k < kEPT; ++k) {
    const long i = EPT_INDEX(k);
    if (i < n) x[i] = a;
  }
}

// z may alias x or y (pointwiseMult(invD, y, y) in the Chebyshev power method):
// each element is read and written by the same lane, so aliasing is harmless.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_pmult(int n, const T* x, const T* y, T* z) {
#pragma unroll
  for (int k = 0; k < kEPT; ++k) {
    const long i = EPT_INDEX(k);
    if (i < n) z[i] = x[i] * y[i];
  }
}

// The launch's total by its last workgroup, by the tree of the finalize (reduce.hip: 1024 lanes, lane t takes
// partials t, t + 1024, ..). Up to kOneLaunchBlocks workgroups a
// reduction is finished in its own launch: 1.3 us less a dot product than with the finalize's launch up to 768
// workgroups (an axpy and two dots: 16.3 -> 13.5 us), as much at 1024 (16.3 against 16.2), where the arrivals take as long.
constexpr int kOneLaunchBlocks = kTicketGroup * kTicketGroups;
__device__ __forceinline__ void finish_one(double partial, RedWork w, double* out, HostPost post) {
  constexpr int kFinLanes = 1024, U = kFinLanes / kBlock;
  __shared__ double lds[kFinLanes / kWave];
  if (threadIdx.x == 0) __hip_atomic_store(w.partial + blockIdx.x, partial, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (!last_block(w.ticket)) return;
  const int nblk = gridDim.x;
  double p[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int b = u * kBlock + threadIdx.x;
    p[u] = b < nblk ? 0.0 + __hip_atomic_load(w.partial + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const double s = wave_total(p[u]);
    if ((threadIdx.x & (kWave - 1)) == 0) lds[u * (kBlock / kWave) + threadIdx.x / kWave] = s;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  double t = 0.0;
#pragma unroll
  for (int q = 0; q < kFinLanes / kWave; ++q) t += lds[q];
  if (post.to) post_double(post, t);
  out[0] = t;
}

// ONE: finished by its last workgroup, else the partials are left to a finalize
template <typename T, bool ONE>
__global__ void __launch_bounds__(kBlock) k_dot(int n, const T* __restrict__ x, const T* __restrict__ y,
                                                 RedWork w, double* out, HostPost post) {
  __shared__ double lds4[4];
  T xv[kEPT], yv[kEPT];
#pragma unroll
  for (int k = 0; k < kEPT; ++k) {
    const long i = EPT_INDEX(k);
    xv[k] = (i < n) ? x[i] : T(0);
    yv[k] = (i < n) ? y[i] : T(0);
  }
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < kEPT; ++k) s += (double)xv[k] * (double)yv[k];
  double v[1] = {block_sum(s, lds4)};
  if constexpr (ONE) finish_one(v[0], w, out, post);
  else store_partials<1>(v, w);
}

// y += a x ; out = y . y
template <typename T, bool ONE>
__global__ void __launch_bounds__(kBlock) k_axpy_dot(int n, T a, const T* __restrict__ x, T* __restrict__ y,
                                                      RedWork w, double* out) {
  __shared__ double lds4[4];
  T xv[kEPT], yv[kEPT];
#pragma unroll
  for (int k = 0; k < kEPT; ++k) {
    const long i = EPT_INDEX(k);
    xv[k] = (i < n) ? x[i] : T(0);
    yv[k] = (i < n) ? y[i] : T(0);
  }
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < kEPT; ++k) {
    const long i = EPT_INDEX(k);
    const T v = yv[k] + a * xv[k];
    if (i < n) {
      y[i] = v;
      s += (double)v * (double)v;
    }
  }
  double v[1] = {block_sum(s, lds4)};
  if constexpr (ONE) finish_one(v[0], w, out, HostPost{});
  else store_partials<1>(v, w);
}

// ---- launchers --------------------------------------------------------------
static inline dim3 ept_grid(long n) { return dim3((unsigned)ept_blocks(n)); }

template <typename T>
void launch_copy(hipStream_t st, int n, const T* x, T* y) {
  if (n > 0) hipLaunchKernelGGL(k_copy<T>, ept_grid(n), dim3(kBlock), 0, st, n, x, y);
}
template <typename T>
void launch_axpy(hipStream_t st, int n, T a, const T* x, T* y) {
  if (n > 0) hipLaunchKernelGGL(k_axpy<T>, ept_grid(n), dim3(kBlock), 0, st, n, a, x, y);
}
template <typename T>
void launch_scal(hipStream_t st, int n, T a, T* x) {
  if (n > 0) hipLaunchKernelGGL(k_scal<T>, ept_grid(n), dim3(kBlock), 0, st, n, a, x);
}
template <typename T>
void launch_assign(hipStream_t st, int n, T a, T* x) {
  if (n > 0) hipLaunchKernelGGL(k_assign<T>, ept_grid(n), dim3(kBlock), 0, st, n, a, x);
}
template <typename T>
void launch_pmult(hipStream_t st, int n, const T* x, const T* y, T* z) {
  if (n > 0) hipLaunchKernelGGL(k_pmult<T>, ept_grid(n), dim3(kBlock), 0, st, n, x, y, z);
}
template <typename T>
void launch_dot(hipStream_t st, RedWork w, int n, const T* x, const T* y, double* out, HostPost post) {
  if (w.ticket && ept_blocks(n) <= kOneLaunchBlocks) {
    hipLaunchKernelGGL((k_dot<T, true>), ept_grid(n), dim3(kBlock), 0, st, n, x, y, w, out, post);
    return;
  }
  hipLaunchKernelGGL((k_dot<T, false>), ept_grid(n), dim3(kBlock), 0, st, n, x, y, w, out, post);
  if (post.to) launch_finalize_post(st, w, ept_blocks(n), out, post);
  else launch_finalize(st, w, ept_blocks(n), 1, kFinStore, out, nullptr);
}
template <typename T>
void launch_axpy_dot(hipStream_t st, RedWork w, int n, T a, const T* x, T* y, double* out) {
  if (w.ticket && ept_blocks(n) <= kOneLaunchBlocks) {
    hipLaunchKernelGGL((k_axpy_dot<T, true>), ept_grid(n), dim3(kBlock), 0, st, n, a, x, y, w, out);
    return;
  }
  hipLaunchKernelGGL((k_axpy_dot<T, false>), ept_grid(n), dim3(kBlock), 0, st, n, a, x, y, w, out);
  launch_finalize(st, w, ept_blocks(n), 1, kFinStore, out, nullptr);
}

#define ALIEN_HIP_INST_BLAS1(T)                                                         \
  template void launch_copy<T>(hipStream_t, int, const T*, T*);                         \
  template void launch_axpy<T>(hipStream_t, int, T, const T*, T*);                      \
  template void launch_scal<T>(hipStream_t, int, T, T*);                                \
  template void launch_assign<T>(hipStream_t, int, T, T*);                              \
  template void launch_pmult<T>(hipStream_t, int, const T*, const T*, T*);              \
  template void launch_dot<T>(hipStream_t, RedWork, int, const T*, const T*, double*, HostPost); \
  template void launch_axpy_dot<T>(hipStream_t, RedWork, int, T, const T*, T*, double*);
ALIEN_HIP_INST_BLAS1(double)
ALIEN_HIP_INST_BLAS1(float)

// y[k] = x[idx[k]]: the values of a permuted copy of a matrix
__global__ void __launch_bounds__(kBlock) k_gather_f64(long n, const int* __restrict__ idx,
                                                        const double* __restrict__ x, double* __restrict__ y) {
  const long i = blockIdx.x * (long)kBlock + threadIdx.x;
  if (i < n) y[i] = x[idx[i]];
}
void launch_gather_f64(hipStream_t st, long n, const int* idx, const double* x, double* y) {
  if (n > 0)
    hipLaunchKernelGGL(k_gather_f64, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, n, idx, x, y);
}

} // namespace alien_hip
