// Learned preconditioner M = G G^T: graph network forward, backward, losses and
// optimiser on gfx950 (no counterpart in the reference; see the oracle's
// statement of the model in oracle/gnn_oracle.py for the mathematics).
//
// Model, for an SPD matrix A with a symmetric pattern (d_i = a_ii):
//   e_ij = -a_ij / sqrt(d_i d_j),  f_i = [1, s_i, 1 - s_i, max_j e_ij],  s_i = sum_j e_ij
//   h0 = relu(f W_in + b_in)                                      (N x 32)
//   h_l = h_{l-1} + relu([h_{l-1}, E h_{l-1}] W_l + b_l)   l = 1..3
//   Ghat_ii = exp(h3_i . w_d + c_d),  Ghat_ij = e_ij (h3_i . w_a + h3_j . w_b + c_e)  (j < i)
//   G = D^-1/2 Ghat,  M = G G^T
// Dense layers run on the matrix cores: v_mfma_f32_32x32x8_bf16 with bf16
// weights and bf16-rounded inputs, FP32 accumulation. Every reduction over
// rows (losses, weight gradients) uses per-workgroup partials summed in a fixed
// order: the results are deterministic.
#include <hip/hip_runtime.h>

#include <array>
#include <cmath>
#include <vector>

#include "../alien_hip_internal.h"
#include "device_common.h"
#include "gnn.h"
#include "launch.h"
#include "wave_total.h"

namespace alien_hip {
namespace gnn {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// float -> bfloat16 bits, round to nearest even (NaN stays NaN, quieted). Branch-free: both
// results are formed and one selected (v_cndmask), where an early return for NaN made every
// conversion a divergent branch and left the dense layers' operand conversion instruction-bound.
__device__ __forceinline__ short to_bf16(float x) {
  const unsigned u = __float_as_uint(x);
  const unsigned rounded = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
  const unsigned quiet = (u >> 16) | 0x40u;
  return (short)((u & 0x7fffffffu) > 0x7f800000u ? quiet : rounded);
}
__device__ __forceinline__ float bf16_round(float x) {
  return __uint_as_float(((unsigned)(unsigned short)to_bf16(x)) << 16);
}

// ---- graph preparation ----------------------------------------------------------------
__global__ void k_prep_dis(int n, const int* __restrict__ dcol, const double* __restrict__ vals,
                           float* __restrict__ dis) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dis[i] = (float)(1.0 / sqrt(vals[dcol[i]]));
}
// e per CSR entry (0 on the diagonal) and the node features
__global__ void k_prep_feat(int n, const int* __restrict__ ro, const int* __restrict__ cols,
                            const double* __restrict__ vals, const float* __restrict__ dis, float* __restrict__ e,
                            float* __restrict__ f) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.f, mx = 0.f, up = 0.f, lo = 0.f;
  bool any = false;
  for (int k = ro[i]; k < ro[i + 1]; ++k) {
    const int j = cols[k];
    float v = 0.f;
    if (j != i) {
      v = (float)(-vals[k] * (double)dis[i] * (double)dis[j]);
      s += v;
      mx = any ? fmaxf(mx, v) : v;
      any = true;
      if (j > i) up += v * v;
      else lo += v * v;
    }
    e[k] = v;
  }
  float* fi = f + (long)i * kFeat;
  fi[0] = 1.f;
  fi[1] = s;
  fi[2] = 1.f - s;
  fi[3] = mx;
  fi[4] = up;
  fi[5] = lo;
}

// ---- dense layer on MFMA --------------------------------------------------------------------
// Z = [X0 | X1] W + b ; H = Hres + relu(Z)   (Hres may be NULL: H = relu(Z))
// X0 holds input columns [0, c0), X1 columns [c0, kin); kin <= KIN (multiple of 8).
// One wavefront computes 32 rows x 32 outputs: KIN/8 mfma 32x32x8 steps.
// Lane l holds A[row = l%32][k = 4(l/32)..+3], B[k][col = l%32], and the result
// D[8 (r/4) + 4 (l/32) + r%4][l%32] in accumulator register r.
//
// Message-passing layers (KIN = 64: X0 = h, X1 = m, both n x 32, Hres = h): each wave first copies
// its 32 rows of h and m into LDS with 16-byte loads (a contiguous 4 KB block each), then reads
// the MFMA operands and the residual term from there: h is read from memory once, not twice, and
// the row-strided 4-byte operand loads become coalesced 16-byte ones. Same values, same MFMA
// sequence: the results are those of the direct form below.
constexpr int kDenseLdsPitch = 2 * kHidden + 1; // one pad float: the 32 rows of a column hit 32 banks
template <int KIN>
__global__ void __launch_bounds__(256) k_dense(int n, const float* __restrict__ X0, int ld0, int c0,
                                               const float* __restrict__ X1, int ld1, int kin,
                                               const float* __restrict__ W, const float* __restrict__ b,
                                               const float* __restrict__ Hres, float* __restrict__ Z,
                                               float* __restrict__ Hout) {
  const int lane = threadIdx.x & 63;
  const int wave = (blockIdx.x * 256 + threadIdx.x) >> 6;
  const int r0 = wave * 32;
  const int kb = lane >> 5;
  const int col = lane & 31;
  if constexpr (KIN == 2 * kHidden) {
    __shared__ float xs[4][32][kDenseLdsPitch];
    const bool staged = ld0 == kHidden && ld1 == kHidden && c0 == kHidden && kin == KIN && (!Hres || Hres == X0);
    if (staged) { // uniform over the grid
      float(*x)[kDenseLdsPitch] = xs[threadIdx.x >> 6];
      // the lane's weights for every step, loaded beside the activations (one round trip for both,
      // where loading them inside the step loop cost a round trip per step)
      float wv[KIN / 8][4];
#pragma unroll
      for (int ks = 0; ks < KIN / 8; ++ks)
#pragma unroll
        for (int v = 0; v < 4; ++v) wv[ks][v] = W[(ks * 8 + kb * 4 + v) * kHidden + col];
      const float bias = b[col];
#pragma unroll
      for (int part = 0; part < 2; ++part) {
        const float* src = part ? X1 : X0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int f = j * 64 + lane; // float4 index in the wave's 32 x 32 block
          const int rr = f >> 3, c4 = (f & 7) * 4;
          float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
          if (r0 + rr < n) v = *reinterpret_cast<const float4*>(src + (long)(r0 + rr) * kHidden + c4);
          float* d = &x[rr][part * kHidden + c4];
          d[0] = v.x;
          d[1] = v.y;
          d[2] = v.z;
          d[3] = v.w;
        }
      }
      __syncthreads(); // every wave reaches it (no early return above)
      if (r0 >= n) return;
      f32x16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KIN / 8; ++ks) {
        bf16x4 a, bb;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          a[v] = to_bf16(x[lane & 31][ks * 8 + kb * 4 + v]);
          bb[v] = to_bf16(wv[ks][v]);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, bb, acc, 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int rl = 8 * (r >> 2) + 4 * kb + (r & 3);
        const int row = r0 + rl;
        if (row < n) {
          const float z = acc[r] + bias;
          const long o = (long)row * kHidden + col;
          if (Z) Z[o] = z;
          Hout[o] = (Hres ? x[rl][col] : 0.f) + fmaxf(z, 0.f);
        }
      }
      return;
    }
  }
  if (r0 >= n) return;
  const int arow = r0 + (lane & 31);
  f32x16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ks = 0; ks < KIN / 8; ++ks) {
    bf16x4 a, bb;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int k = ks * 8 + kb * 4 + v;
      float xa = 0.f, wb = 0.f;
      if (k < kin) {
        if (arow < n) xa = (k < c0) ? X0[(long)arow * ld0 + k] : X1[(long)arow * ld1 + (k - c0)];
        wb = W[k * kHidden + col];
      }
      a[v] = to_bf16(xa);
      bb[v] = to_bf16(wb);
    }
    acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(a, bb, acc, 0, 0, 0);
  }
  const float bias = b[col];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = r0 + 8 * (r >> 2) + 4 * kb + (r & 3);
    if (row < n) {
      const float z = acc[r] + bias;
      const long o = (long)row * kHidden + col;
      if (Z) Z[o] = z;
      Hout[o] = (Hres ? Hres[o] : 0.f) + fmaxf(z, 0.f);
    }
  }
}

// m_i = sum_{j != i} e_ij h_j   (32 lanes per row, one feature per lane)
// 8 lanes per row, 4 features per lane (one 16-byte load of the neighbour's row
// chunk), 32 rows per workgroup; workgroups are remapped so that each XCD takes
// chunks of consecutive rows (its L2 then holds the x- and y-neighbours' rows).
// Per feature the sum runs over the row's entries in order, as one lane per feature.
constexpr int kAggRows = 32;
constexpr int kAggChunk = 64;
__global__ void __launch_bounds__(256) k_aggregate(int n, const int* __restrict__ ro, const int* __restrict__ cols,
                                                   const float* __restrict__ e, const float* __restrict__ h,
                                                   float* __restrict__ m) {
  const int p = blockIdx.x, q = p / kXcds;
  const int logical = (q / kAggChunk) * (kXcds * kAggChunk) + (p % kXcds) * kAggChunk + q % kAggChunk;
  const int i = logical * kAggRows + (threadIdx.x >> 3);
  const int c4 = threadIdx.x & 7;
  if (i >= n) return;
  float4 acc = {0.f, 0.f, 0.f, 0.f};
  const float4* __restrict__ h4 = reinterpret_cast<const float4*>(h);
  for (int k = ro[i]; k < ro[i + 1]; ++k) {
    const float w = e[k];
    if (w != 0.f) {
      const float4 v = h4[(long)cols[k] * (kHidden / 4) + c4];
      acc.x += w * v.x;
      acc.y += w * v.y;
      acc.z += w * v.z;
      acc.w += w * v.w;
    }
  }
  reinterpret_cast<float4*>(m)[(long)i * (kHidden / 4) + c4] = acc;
}
inline dim3 aggregate_grid(int n) {
  const long g = (n + kAggRows - 1) / kAggRows;
  const long q = (long)kXcds * kAggChunk;
  return dim3((unsigned)((g + q - 1) / q * q));
}

// ---- output head ------------------------------------------------------------------------------
__device__ __forceinline__ float dot32(const float* __restrict__ a, const float* __restrict__ w) {
  float s = 0.f;
#pragma unroll
  for (int q = 0; q < kHidden; ++q) s += a[q] * w[q];
  return s;
}

// ghat per CSR entry: diagonal exp(h_i.w_d + c_d), strictly lower e_ij (h_i.w_a + h_j.w_b + c_e),
// upper entries 0 (G is lower triangular)
__global__ void k_head(int n, const int* __restrict__ ro, const int* __restrict__ cols, const int* __restrict__ dcol,
                       const float* __restrict__ e, const float* __restrict__ h, const float* __restrict__ P,
                       float* __restrict__ ghat) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float* hi = h + (long)i * kHidden;
  const float ai = dot32(hi, P + kOffWa);
  ghat[dcol[i]] = expf(dot32(hi, P + kOffWd) + P[kOffCd]);
  for (int k = ro[i]; k < dcol[i]; ++k) {
    const float* hj = h + (long)cols[k] * kHidden;
    ghat[k] = e[k] * (ai + dot32(hj, P + kOffWb) + P[kOffCe]);
  }
  for (int k = dcol[i] + 1; k < ro[i + 1]; ++k) ghat[k] = 0.f;
}

// ---- losses ------------------------------------------------------------------------------------
// Kaporin term. For each lower entry (i,j) of Ghat: AG_ij = sum_k Ahat_ik Ghat_kj,
// Ahat_ik = 1 (k = i) or -e_ik; Ghat_kj read at the position of column j in row k.
__device__ __forceinline__ int find_col(const int* __restrict__ cols, int b, int e, int j) {
  for (int k = b; k < e; ++k)
    if (cols[k] == j) return k;
  return -1;
}
// The gradient uses the symmetric part, ((A + A^T) Ghat)_ij / 2, read through the
// transpose positions (A^T)_ic = A_ci = -e at tpos (equal to AG for symmetric A).
__global__ void __launch_bounds__(256) k_kcond(int n, const int* __restrict__ ro, const int* __restrict__ cols,
                                               const int* __restrict__ dcol, const int* __restrict__ tpos,
                                               const float* __restrict__ e, const float* __restrict__ ghat,
                                               float* __restrict__ ag, RedWork w) {
  __shared__ double lds[4];
  double tr = 0.0, ld = 0.0;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
    for (int p = ro[i]; p <= dcol[i]; ++p) { // lower entries and the diagonal of row i
      const int j = cols[p];
      float s = 0.f, st = 0.f;
      for (int k2 = ro[i]; k2 < ro[i + 1]; ++k2) {
        const int c = cols[k2];
        if (c < j) continue;                       // Ghat_cj = 0 above the diagonal
        const int q = find_col(cols, ro[c], dcol[c] + 1, j); // (c, j) in c's lower part
        if (q < 0) continue;
        const float a = (c == i) ? 1.f : -e[k2];
        const float at = (c == i) ? 1.f : -e[tpos[k2]];
        s += a * ghat[q];
        st += at * ghat[q];
      }
      ag[p] = 0.5f * (s + st);
      tr += (double)ghat[p] * (double)s;
    }
    ld = log((double)ghat[dcol[i]]);
  }
  double v[2];
  v[0] = block_sum(tr, lds);
  __syncthreads();
  v[1] = block_sum(ld, lds);
  store_partials<2>(v, w);
}

// probe term, K probes stored row-major (N x K)
template <int K>
__global__ void k_ahat_mult(int n, const int* __restrict__ ro, const int* __restrict__ cols, const float* __restrict__ e,
                            const float* __restrict__ V, float* __restrict__ W) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float acc[K];
#pragma unroll
  for (int c = 0; c < K; ++c) acc[c] = 0.f;
  for (int k = ro[i]; k < ro[i + 1]; ++k) {
    const int j = cols[k];
    const float a = (j == i) ? 1.f : -e[k];
#pragma unroll
    for (int c = 0; c < K; ++c) acc[c] += a * V[(long)j * K + c];
  }
#pragma unroll
  for (int c = 0; c < K; ++c) W[(long)i * K + c] = acc[c];
}
// Y = Ghat X (lower rows) or Y = Ghat^T X (upper rows through the transpose positions)
template <int K, bool TRANS>
__global__ void k_ghat_mult(int n, const int* __restrict__ ro, const int* __restrict__ cols, const int* __restrict__ dcol,
                            const int* __restrict__ tpos, const float* __restrict__ ghat, const float* __restrict__ X,
                            float* __restrict__ Y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float acc[K];
#pragma unroll
  for (int c = 0; c < K; ++c) acc[c] = 0.f;
  const int b = TRANS ? dcol[i] : ro[i];
  const int en = TRANS ? ro[i + 1] : dcol[i] + 1;
  for (int k = b; k < en; ++k) {
    const int j = cols[k];
    const float g = TRANS ? ghat[tpos[k]] : ghat[k];
#pragma unroll
    for (int c = 0; c < K; ++c) acc[c] += g * X[(long)j * K + c];
  }
#pragma unroll
  for (int c = 0; c < K; ++c) Y[(long)i * K + c] = acc[c];
}
// R = V - Y, dY = -2 R / (N K), loss partial sum R^2
template <int K>
__global__ void __launch_bounds__(256) k_probe_resid(int n, const float* __restrict__ V, const float* __restrict__ Y,
                                                     float* __restrict__ dY, float scale, RedWork w) {
  __shared__ double lds[4];
  double s = 0.0;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) {
#pragma unroll
    for (int c = 0; c < K; ++c) {
      const float r = V[(long)i * K + c] - Y[(long)i * K + c];
      dY[(long)i * K + c] = -2.f * r * scale;
      s += (double)r * (double)r;
    }
  }
  double v[1] = {block_sum(s, lds)};
  store_partials<1>(v, w);
}

// ---- dL/dGhat -> dL/d(head inputs) --------------------------------------------------------------
// g_ij (per lower CSR entry) = kw (2 AG_ij / tr - (2/N) [i==j] / Ghat_ii) + beta (sum_c dY_ic U_jc + W_ic Q_jc)
template <int K>
__global__ void k_grad_ghat(int n, const int* __restrict__ ro, const int* __restrict__ cols, const int* __restrict__ dcol,
                            const float* __restrict__ ghat, const float* __restrict__ ag, const double* __restrict__ sums,
                            float kw, float beta, const float* __restrict__ dY, const float* __restrict__ U,
                            const float* __restrict__ Wp, const float* __restrict__ Q, float* __restrict__ gg) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float tr = kw != 0.f ? (float)sums[0] : 1.f;
  for (int k = ro[i]; k <= dcol[i]; ++k) {
    const int j = cols[k];
    float g = 0.f;
    if (kw != 0.f) {
      g = 2.f * ag[k] / tr;
      if (k == dcol[i]) g -= 2.f / ((float)n * ghat[k]);
      g *= kw;
    }
    if (beta != 0.f) {
      float p = 0.f;
#pragma unroll
      for (int c = 0; c < K; ++c) p += dY[(long)i * K + c] * U[(long)j * K + c] + Wp[(long)i * K + c] * Q[(long)j * K + c];
      g += beta * p;
    }
    gg[k] = g;
  }
}

// ---- k-step CG loss (N x 4 column blocks, one right-hand side per column) ----
struct Coef4 {
  float c[4];
};

// Three launches a step forward, three in the reverse pass. One lane per row, its four columns in one 16-byte value.
// Each element is computed by the operations and in the order of the separate products, dots and combinations it
// stands for, a neighbour's element that has not been stored yet by the same operations again: the results do not
// depend on the fusion. Step scalars stay on the device: a kernel that needs a dot product finalizes the partials of
// the launch before (up to one wavefront's lanes of them; larger systems launch the finalize and read one total), and
// its first workgroup keeps the value for later steps. When the host read every dot product back (64 of them on a
// 16^3 system with 16 steps) and a step took 23 launches, that gradient took 3.70 ms; now 1.04. Dependent loads and
// launch latency bound a launch: 3.9 us (products alone) to 6.5 (with a scalar to finalize first).
struct Dot4 {
  const double* p; // value c's partials at p[c * n ..)
  int n;           // at most kWave
};
// the total of column lane % 4 (every lane of the wavefront calls it)
__device__ __forceinline__ double dot_value(Dot4 d) {
  const int lane = threadIdx.x & (kWave - 1);
  double in[4], v[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) in[c] = lane < d.n ? 0.0 + d.p[c * d.n + lane] : 0.0;
#pragma unroll
  for (int c = 0; c < 4; ++c) v[c] = 0.0 + wave_total(in[c]);
  return lane & 2 ? (lane & 1 ? v[3] : v[2]) : (lane & 1 ? v[1] : v[0]);
}
// column lane % 4 of a kept scalar
__device__ __forceinline__ double kept(const double* s) { return s[threadIdx.x & 3]; }
__device__ __forceinline__ void keep(double* to, double v) {
  if (blockIdx.x == 0 && threadIdx.x < 4) to[threadIdx.x] = v;
}
// the four columns' values of v, held by lanes 0..3
__device__ __forceinline__ void columns(double v, float (&to)[4]) {
  const int f = __float_as_int((float)v);
#pragma unroll
  for (int c = 0; c < 4; ++c) to[c] = __int_as_float(__builtin_amdgcn_readlane(f, c));
}
// per-column partials of X . Y of this workgroup's rows at part[c * stride + workgroup] (block_sum's tree,
// the four columns in one pass); lds: 16 doubles, not read or written by the workgroup otherwise
__device__ __forceinline__ void dot_partials(bool in, const float4& X, const float4& Y, double* part, int stride,
                                             double* lds) {
  const float x[4] = {X.x, X.y, X.z, X.w}, y[4] = {Y.x, Y.y, Y.z, Y.w};
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const double s = wave_total(in ? (double)x[c] * (double)y[c] : 0.0);
    if (lane == 0) lds[c * 4 + wave] = s;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double r = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) r += lds[threadIdx.x * 4 + q];
    part[(long)threadIdx.x * stride + blockIdx.x] = r;
  }
}
__device__ __forceinline__ float4 axpy4(float4 x, const float (&b)[4], float4 z) { // 1 x + b z
  return make_float4(x.x + b[0] * z.x, x.y + b[1] * z.y, x.z + b[2] * z.z, x.w + b[3] * z.w);
}
__device__ __forceinline__ float4 scale4(const float (&a)[4], float4 x) {
  return make_float4(a[0] * x.x, a[1] * x.y, a[2] * x.z, a[3] * x.w);
}
__device__ __forceinline__ float4 add4(float4 x, float4 y) { return make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w); }
__device__ __forceinline__ void mac4(float4& acc, float g, float4 v) {
  acc.x += g * v.x;
  acc.y += g * v.y;
  acc.z += g * v.z;
  acc.w += g * v.w;
}
struct CgRows { // the system and the factor
  int n;
  const int *ro, *cols, *dcol, *tpos;
  const float *e, *ghat;
};
// Sum over the entries [b, e) of a row (b < e), in order, of coefficient(entry, column) * use(load(column)).
// kBatch entries' columns are loaded together, then their coefficients and vectors; ready() is called
// once, by every lane, with the first of these loads in flight: it waits for the step's scalars.
// (One entry after the other, behind the scalars, took two or three round trips to memory an entry.)
constexpr int kBatch = 8;
template <typename C, typename L, typename R, typename U>
__device__ __forceinline__ float4 row_sum(const int* __restrict__ cols, int b, int e, C coef, L load, R ready, U use) {
  int j[kBatch];
  float a[kBatch];
  decltype(load(0)) v[kBatch];
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  auto fetch = [&] {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) j[u] = cols[min(b + u, e - 1)];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) a[u] = coef(min(b + u, e - 1), j[u]);
#pragma unroll
    for (int u = 0; u < kBatch; ++u) v[u] = load(j[u]);
  };
  auto add = [&] {
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (b + u < e) mac4(acc, a[u], use(v[u]));
  };
  fetch();
  ready();
  add();
  for (b += kBatch; b < e; b += kBatch) {
    fetch();
    add();
  }
  return acc;
}
// rows of Ahat, Ghat and Ghat^T
template <typename L, typename R, typename U>
__device__ __forceinline__ float4 ahat_row(const CgRows& A, int i, L load, R ready, U use) {
  return row_sum(A.cols, A.ro[i], A.ro[i + 1], [&](int k, int j) { return j == i ? 1.f : -A.e[k]; }, load, ready, use);
}
template <typename L, typename R, typename U>
__device__ __forceinline__ float4 ghat_row(const CgRows& A, int i, L load, R ready, U use) {
  return row_sum(A.cols, A.ro[i], A.dcol[i] + 1, [&](int k, int) { return A.ghat[k]; }, load, ready, use);
}
template <typename L, typename R, typename U>
__device__ __forceinline__ float4 ghat_t_row(const CgRows& A, int i, L load, R ready, U use) {
  return row_sum(A.cols, A.dcol[i], A.ro[i + 1], [&](int k, int) { return A.ghat[A.tpos[k]]; }, load, ready, use);
}
struct Two4 {
  float4 x, y;
};
// this lane's row; lanes past the last one work on it again and store nothing
struct CgLane {
  bool in;
  int i;
  __device__ __forceinline__ explicit CgLane(int n) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    in = t < n;
    i = min(t, n - 1);
  }
};
#define CG4_PLAIN [] {}, [](float4 v) { return v; }

// T = Ghat^T R with T.T and R.R
__global__ void __launch_bounds__(256) k_cg4_start(CgRows A, const float4* __restrict__ R, float4* __restrict__ T,
                                                   double* tt, double* rr, int stride) {
  __shared__ double lds[32];
  const CgLane me(A.n);
  const float4 r = R[me.i];
  const float4 t = ghat_t_row(A, me.i, [&](int j) { return R[j]; }, CG4_PLAIN);
  if (me.in) T[me.i] = t;
  dot_partials(me.in, t, t, tt, stride, lds);
  dot_partials(me.in, r, r, rr, stride, lds + 16);
}
// P = Ghat T, or P = Ghat T + (rho1 / rho) P0; keeps rho1
__global__ void __launch_bounds__(256) k_cg4_dir(CgRows A, const float4* __restrict__ T, const float4* __restrict__ P0,
                                                 Dot4 rho1, const double* __restrict__ rho, double* keep_rho1,
                                                 float4* __restrict__ P) {
  const CgLane me(A.n);
  float4 p0 = make_float4(0.f, 0.f, 0.f, 0.f);
  double r0 = 1.0;
  if (P0) {
    p0 = P0[me.i];
    r0 = kept(rho);
  }
  float b[4];
  const float4 z = ghat_row(A, me.i, [&](int j) { return T[j]; },
                            [&] {
                              const double r1 = dot_value(rho1);
                              keep(keep_rho1, r1);
                              columns(r1 / r0, b);
                            },
                            [](float4 v) { return v; });
  if (me.in) P[me.i] = P0 ? axpy4(z, b, p0) : z;
}
// Q = Ahat P with P.Q
__global__ void __launch_bounds__(256) k_cg4_ap(CgRows A, const float4* __restrict__ P, float4* __restrict__ Q,
                                                double* pq, int stride) {
  __shared__ double lds[16];
  const CgLane me(A.n);
  const float4 p = P[me.i];
  const float4 q = ahat_row(A, me.i, [&](int j) { return P[j]; }, CG4_PLAIN);
  if (me.in) Q[me.i] = q;
  dot_partials(me.in, p, q, pq, stride, lds);
}
// R1 = R - (rho / sig) Q; T1 = Ghat^T R1 with T1.T1, or (T1 NULL) R1.R1; keeps sig
__global__ void __launch_bounds__(256) k_cg4_res(CgRows A, const float4* __restrict__ R, const float4* __restrict__ Q,
                                                 const double* __restrict__ rho, Dot4 sig, double* keep_sig,
                                                 float4* __restrict__ R1, float4* __restrict__ T1, double* dot,
                                                 int stride) {
  __shared__ double lds[16];
  const CgLane me(A.n);
  const float4 r0 = R[me.i], q0 = Q[me.i];
  const double rh = kept(rho);
  float na[4];
  auto scalars = [&] {
    const double sg = dot_value(sig);
    keep(keep_sig, sg);
    columns(-(rh / sg), na);
  };
  float4 d;
  if (T1) {
    d = ghat_t_row(A, me.i, [&](int j) { return Two4{R[j], Q[j]}; }, scalars,
                   [&](Two4 v) { return axpy4(v.x, na, v.y); });
    if (me.in) T1[me.i] = d;
  } else {
    scalars();
  }
  const float4 r = axpy4(r0, na, q0);
  if (me.in) R1[me.i] = r;
  if (!T1) d = r;
  dot_partials(me.in, d, d, dot, stride, lds);
}
// reverse: rbar = (2 / (4 rrk)) R with Q.rbar
__global__ void __launch_bounds__(256) k_cg4_rev_start(int n, Coef4 c0, const float4* __restrict__ R,
                                                       const float4* __restrict__ Q, float4* __restrict__ rbar,
                                                       double* qr, int stride) {
  __shared__ double lds[16];
  const CgLane me(n);
  const float4 r = scale4(c0.c, R[me.i]), q = Q[me.i];
  if (me.in) rbar[me.i] = r;
  dot_partials(me.in, q, r, qr, stride, lds);
}
// z = Ghat t, rho = t.t: tbar = 2 rhobar T + Ghat^T pbar, with rhobar = rhobar_next + betabar / rho (or
// rhobar_next alone: rho NULL); keeps what rho's own adjoint takes from beta, -betabar rho1 / rho^2
__global__ void __launch_bounds__(256) k_cg4_rev_t(CgRows A, const float4* __restrict__ pbar, const float4* __restrict__ T,
                                                   const double* __restrict__ rhobar_next, Dot4 betabar,
                                                   const double* __restrict__ rho, const double* __restrict__ rho1,
                                                   double* keep_own, float4* __restrict__ tbar) {
  const CgLane me(A.n);
  const float4 own = T[me.i];
  float two[4];
  const float4 t = ghat_t_row(A, me.i, [&](int j) { return pbar[j]; },
                              [&] {
                                double rb = kept(rhobar_next);
                                if (rho) {
                                  const double r = kept(rho), r1 = kept(rho1), bb = dot_value(betabar);
                                  rb = rb + bb / r;
                                  keep(keep_own, 0.0 - bb * r1 / (r * r));
                                }
                                columns(2.0 * rb, two);
                              },
                              [](float4 v) { return v; });
  if (me.in) tbar[me.i] = add4(scale4(two, own), t);
}
// t = Ghat^T r, z = Ghat t: dL/dGhat += pbar T^T + R tbar^T over the lower pattern; rbar += Ghat tbar
// with Q.rbar (rbar NULL: the first residual, fixed)
__global__ void __launch_bounds__(256) k_cg4_rev_r(CgRows A, const float4* __restrict__ pbar, const float4* __restrict__ T,
                                                   const float4* __restrict__ R, const float4* __restrict__ tbar,
                                                   float* __restrict__ gg, float4* __restrict__ rbar,
                                                   const float4* __restrict__ Q, double* qr, int stride) {
  __shared__ double lds[16];
  constexpr int kHalf = kBatch / 2; // two vectors an entry
  const CgLane me(A.n);
  const float4 u = pbar[me.i], w = R[me.i];
  float4 r = make_float4(0.f, 0.f, 0.f, 0.f), q = r, acc = r;
  if (rbar) {
    r = rbar[me.i];
    q = Q[me.i];
  }
  const int e = A.dcol[me.i] + 1;
  for (int k = A.ro[me.i]; k < e; k += kHalf) {
    float4 v[kHalf], x[kHalf];
    float g[kHalf], old[kHalf];
#pragma unroll
    for (int m = 0; m < kHalf; ++m) {
      const int km = min(k + m, e - 1), l = A.cols[km];
      v[m] = T[l];
      x[m] = tbar[l];
      g[m] = A.ghat[km];
      old[m] = gg[km];
    }
#pragma unroll
    for (int m = 0; m < kHalf; ++m) {
      if (k + m >= e) continue;
      float s = 0.f;
      s += u.x * v[m].x;
      s += w.x * x[m].x;
      s += u.y * v[m].y;
      s += w.y * x[m].y;
      s += u.z * v[m].z;
      s += w.z * x[m].z;
      s += u.w * v[m].w;
      s += w.w * x[m].w;
      if (me.in) gg[k + m] = old[m] + s;
      mac4(acc, g[m], x[m]);
    }
  }
  if (!rbar) return;
  r = add4(r, acc);
  if (me.in) rbar[me.i] = r;
  dot_partials(me.in, q, r, qr, stride, lds);
}
// r1 = r - alpha q, q = Ahat p: qbar = -alpha rbar + sigbar P; pbar = (beta pbar + sigbar Q) + Ahat qbar (beta =
// rho1 / rho; rho1 NULL: no direction follows) with pbar.P0; keeps rhobar = own + alphabar / sig (alphabar = -Q.rbar)
__global__ void __launch_bounds__(256) k_cg4_rev_p(CgRows A, const float4* __restrict__ rbar, const float4* __restrict__ P,
                                                   const float4* __restrict__ Q, const double* __restrict__ rho,
                                                   const double* __restrict__ rho1, const double* __restrict__ sig,
                                                   Dot4 qr, const double* __restrict__ own, double* keep_rhobar,
                                                   float4* __restrict__ pbar, const float4* __restrict__ P0,
                                                   double* betabar, int stride) {
  __shared__ double lds[16];
  const CgLane me(A.n);
  float4 p = make_float4(0.f, 0.f, 0.f, 0.f), p0 = p;
  const float4 q = Q[me.i];
  const double r0 = kept(rho), sg = kept(sig);
  double r1 = 0.0, ow = 0.0;
  if (rho1) {
    r1 = kept(rho1);
    ow = kept(own);
    p = pbar[me.i];
  }
  if (P0) p0 = P0[me.i];
  float na[4], sb[4], be[4];
  const float4 t = ahat_row(A, me.i, [&](int j) { return Two4{rbar[j], P[j]}; },
                            [&] {
                              const double alphabar = -dot_value(qr);
                              keep(keep_rhobar, ow + alphabar / sg);
                              columns(-alphabar * r0 / (sg * sg), sb);
                              columns(-(r0 / sg), na);
                              columns(r1 / r0, be);
                            },
                            [&](Two4 v) { return add4(scale4(na, v.x), scale4(sb, v.y)); });
  if (rho1) p = scale4(be, p);
  p = add4(axpy4(p, sb, q), t);
  if (me.in) pbar[me.i] = p;
  if (P0) dot_partials(me.in, p, p0, betabar, stride, lds);
}
#undef CG4_PLAIN

// head backward: do_i = g_ii ghat_ii, dc_ij = g_ij e_ij;
// dh_i = do_i w_d + sum_{j<i} dc_ij w_a + sum_{m>i} dc_mi w_b ; per-row parameter-gradient terms
// for (w_d, c_d, w_a, w_b, c_e) go to `prow` (N x kHeadGrads) and are summed by k_colsum.
__global__ void k_head_bwd(int n, const int* __restrict__ ro, const int* __restrict__ cols, const int* __restrict__ dcol,
                           const int* __restrict__ tpos, const float* __restrict__ e, const float* __restrict__ ghat,
                           const float* __restrict__ gg, const float* __restrict__ h, const float* __restrict__ P,
                           float* __restrict__ dh, float* __restrict__ prow) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float* hi = h + (long)i * kHidden;
  const float dO = gg[dcol[i]] * ghat[dcol[i]];
  float sa = 0.f, sb = 0.f;      // sum of dc over row i's lower edges / over edges (m, i), m > i
  float wb_acc[kHidden];
#pragma unroll
  for (int q = 0; q < kHidden; ++q) wb_acc[q] = 0.f;
  for (int k = ro[i]; k < dcol[i]; ++k) sa += gg[k] * e[k];
  for (int k = dcol[i] + 1; k < ro[i + 1]; ++k) {
    const int t = tpos[k]; // position of (m, i) in row m, m = cols[k] > i
    const float dc = gg[t] * e[t];
    sb += dc;
    const float* hm = h + (long)cols[k] * kHidden;
#pragma unroll
    for (int q = 0; q < kHidden; ++q) wb_acc[q] += dc * hi[q];
    (void)hm;
  }
  float* pr = prow + (long)i * kHeadGrads;
#pragma unroll
  for (int q = 0; q < kHidden; ++q) {
    dh[(long)i * kHidden + q] = dO * P[kOffWd + q] + sa * P[kOffWa + q] + sb * P[kOffWb + q];
    pr[q] = dO * hi[q];               // w_d
    pr[kHidden + 1 + q] = sa * hi[q]; // w_a: sum over lower edges (i,j) of dc_ij h_i
    pr[2 * kHidden + 1 + q] = wb_acc[q]; // w_b: sum over edges (m,i) of dc_mi h_i
  }
  pr[kHidden] = dO;                    // c_d
  pr[3 * kHidden + 1] = sa;            // c_e (each lower edge counted once, in its row)
}

// dense layer backward (message-passing layers, kin = 64): dz = dh * (z > 0) ; du = dz W^T (W bf16-rounded) ;
// dh_prev = dh + du[:, :32] (the E du[:, 32:] part is added by k_aggregate_add) ; dmsg = du[:, 32:].
// On MFMA: du is a 32-row x 64 x 32 product per wave, 2 output tiles of 16 v_mfma_f32_32x32x2_f32
// steps (FP32 operands: dz and the bf16-rounded weights).
// Each wave stages its 32 rows of dh and dz in LDS (16-byte loads), the workgroup the weights.
__global__ void __launch_bounds__(256) k_dense_bwd_mfma(int n, const float* __restrict__ dh,
                                                        const float* __restrict__ Z, const float* __restrict__ W,
                                                        float* __restrict__ dz, float* __restrict__ dh_prev,
                                                        float* __restrict__ dmsg) {
  __shared__ float ds[4][32][kHidden + 1];
  __shared__ float hs[4][32][kHidden + 1];
  __shared__ float ws[2 * kHidden][kHidden + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r0 = ((blockIdx.x * 256 + threadIdx.x) >> 6) * 32;
  for (int t = threadIdx.x; t < 2 * kHidden * kHidden; t += 256) ws[t / kHidden][t % kHidden] = bf16_round(W[t]);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int f = j * 64 + lane; // float4 index in the wave's 32 x 32 block
    const int rr = f >> 3, c4 = (f & 7) * 4;
    float4 h = make_float4(0.f, 0.f, 0.f, 0.f), z = make_float4(0.f, 0.f, 0.f, 0.f);
    const long o = (long)(r0 + rr) * kHidden + c4;
    if (r0 + rr < n) {
      h = *reinterpret_cast<const float4*>(dh + o);
      z = *reinterpret_cast<const float4*>(Z + o);
    }
    const float4 d = make_float4(z.x > 0.f ? h.x : 0.f, z.y > 0.f ? h.y : 0.f, z.z > 0.f ? h.z : 0.f,
                                 z.w > 0.f ? h.w : 0.f);
    if (r0 + rr < n) *reinterpret_cast<float4*>(dz + o) = d;
    hs[w][rr][c4] = h.x;
    hs[w][rr][c4 + 1] = h.y;
    hs[w][rr][c4 + 2] = h.z;
    hs[w][rr][c4 + 3] = h.w;
    ds[w][rr][c4] = d.x;
    ds[w][rr][c4 + 1] = d.y;
    ds[w][rr][c4 + 2] = d.z;
    ds[w][rr][c4 + 3] = d.w;
  }
  __syncthreads(); // every wave reaches it
  if (r0 >= n) return;
  const int half = lane >> 5, col = lane & 31;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    f32x16 acc = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int qs = 0; qs < kHidden / 2; ++qs) {
      const int q = 2 * qs + half;
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ds[w][col][q], ws[t * kHidden + col][q], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int rl = 8 * (r >> 2) + 4 * half + (r & 3);
      const int row = r0 + rl;
      if (row < n) {
        const long o = (long)row * kHidden + col;
        if (t == 0) dh_prev[o] = hs[w][rl][col] + acc[r];
        else dmsg[o] = acc[r];
      }
    }
  }
}

// dh[i] += sum_{j != i} e_ji dmsg[j]   (E^T dmsg; e_ji read at the transpose position); lanes, rows and
// order of the sums as in k_aggregate (one lane per feature took 563 us at 96^3, this 192)
__global__ void __launch_bounds__(256) k_aggregate_add(int n, const int* __restrict__ ro, const int* __restrict__ cols,
                                                       const int* __restrict__ tpos, const float* __restrict__ e,
                                                       const float* __restrict__ dmsg, float* __restrict__ dh) {
  const int p = blockIdx.x, q = p / kXcds;
  const int logical = (q / kAggChunk) * (kXcds * kAggChunk) + (p % kXcds) * kAggChunk + q % kAggChunk;
  const int i = logical * kAggRows + (threadIdx.x >> 3);
  const int c4 = threadIdx.x & 7;
  if (i >= n) return;
  float4 acc = {0.f, 0.f, 0.f, 0.f};
  const float4* __restrict__ d4 = reinterpret_cast<const float4*>(dmsg);
  for (int k = ro[i]; k < ro[i + 1]; ++k) {
    const float w = e[tpos[k]];
    if (w != 0.f) {
      const float4 v = d4[(long)cols[k] * (kHidden / 4) + c4];
      acc.x += w * v.x;
      acc.y += w * v.y;
      acc.z += w * v.z;
      acc.w += w * v.w;
    }
  }
  float4* __restrict__ to = reinterpret_cast<float4*>(dh) + (long)i * (kHidden / 4) + c4;
  const float4 h = *to;
  *to = make_float4(h.x + acc.x, h.y + acc.y, h.z + acc.z, h.w + acc.w);
}

// Weight-gradient partials: per 256 rows, sum_r bf16(X_r) (x) dz_r  (kin x 32) and sum_r dz_r (32), with
// dz = dz_r where Zm is NULL and dz_r masked by Zm > 0 otherwise.
// Per output FP32 sums of 32 rows, added in FP64 in row order. A workgroup takes COLS of the input columns; the
// KGRP workgroups that share the rows' dz run on one XCD, whose L2 serves it. All 256 rows are loaded at once
// (the loads' latency bounds a small system); then each half-wave sums one chunk of 32 rows, a lane
// a tile of COLS / 4 columns x 4 outputs (1 + COLS / 16 16-byte LDS reads for COLS multiply-adds: one output
// a lane read LDS twice for each and was bound by that on large systems).
// One workgroup for all 64 columns, staging 32 rows at a time, left a 16^3 system's layer on 16 CUs:
// 55 us, 367 at 96^3; this takes 7.1 us at 20^3 and 190 at 96^3.
constexpr int kWgChunk = 32;
// All 64 columns in 8 workgroups of 8 on small systems (latency: 7.2 us against 11.9 at 20^3, 32 row blocks), in 2 of 32 from
// this many row blocks on (dz read twice, not 8 times); 14.4 against 15.0 us at 128 blocks, 20.8 against 20.2 at 250.
constexpr long kWgradWide = 256;
template <int KIN, int COLS>
__global__ void __launch_bounds__(256) k_wgrad_partials(int n, const float* __restrict__ X0, int ld0, int c0,
                                                        const float* __restrict__ X1, int ld1, int kin,
                                                        const float* __restrict__ dz, const float* __restrict__ Zm,
                                                        double* __restrict__ part, int cap) {
  constexpr int KGRP = (KIN + COLS - 1) / COLS;
  constexpr int NCH = 256 / kWgChunk;
  constexpr int KT = COLS / 4;                     // columns of a lane's tile
  constexpr int DCH = kWgChunk * kHidden + kHidden; // floats per chunk, padded: two chunks of a wave on other banks
  constexpr int XCH = kWgChunk * COLS + 32;
  __shared__ __attribute__((aligned(16))) float ds[NCH * DCH];
  __shared__ __attribute__((aligned(16))) float xs[NCH * XCH];
  const int q = blockIdx.x / kXcds;
  const int blk = q / KGRP * kXcds + blockIdx.x % kXcds, k0 = q % KGRP * COLS;
  const int r0 = blk * 256;
  if (r0 >= n) return;
  float4 d[kHidden / 4];
#pragma unroll
  for (int j = 0; j < kHidden / 4; ++j) {
    const int t = j * 256 + threadIdx.x, row = r0 + t / (kHidden / 4);
    const long o = (long)r0 * (kHidden / 4) + t;
    d[j] = row < n ? reinterpret_cast<const float4*>(dz)[o] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (Zm && row < n) {
      const float4 z = reinterpret_cast<const float4*>(Zm)[o];
      d[j] = make_float4(z.x > 0.f ? d[j].x : 0.f, z.y > 0.f ? d[j].y : 0.f, z.z > 0.f ? d[j].z : 0.f,
                         z.w > 0.f ? d[j].w : 0.f);
    }
  }
  float x[COLS];
#pragma unroll
  for (int j = 0; j < COLS; ++j) {
    const int t = j * 256 + threadIdx.x, row = r0 + t / COLS, k = k0 + t % COLS;
    x[j] = row < n && k < kin ? ((k < c0) ? X0[(long)row * ld0 + k] : X1[(long)row * ld1 + (k - c0)]) : 0.f;
  }
#pragma unroll
  for (int j = 0; j < kHidden / 4; ++j) {
    const int t = j * 256 + threadIdx.x, row = t / (kHidden / 4);
    *reinterpret_cast<float4*>(&ds[row / kWgChunk * DCH + row % kWgChunk * kHidden + t % (kHidden / 4) * 4]) = d[j];
  }
#pragma unroll
  for (int j = 0; j < COLS; ++j) {
    const int t = j * 256 + threadIdx.x, row = t / COLS;
    xs[row / kWgChunk * XCH + row % kWgChunk * COLS + t % COLS] = bf16_round(x[j]);
  }
  __syncthreads();
  const int c = threadIdx.x / 32, kq = threadIdx.x % 32 / 8 * KT, jq = threadIdx.x % 8 * 4;
  float s[KT][4], sb[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < KT; ++u)
#pragma unroll
    for (int v = 0; v < 4; ++v) s[u][v] = 0.f;
#pragma unroll 4
  for (int rr = 0; rr < kWgChunk; ++rr) {
    const float4 w = *reinterpret_cast<const float4*>(&ds[c * DCH + rr * kHidden + jq]);
    const float y[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int u = 0; u < KT; ++u) {
      const float xv = xs[c * XCH + rr * COLS + kq + u];
#pragma unroll
      for (int v = 0; v < 4; ++v) s[u][v] += xv * y[v];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) sb[v] += y[v];
  }
  __syncthreads(); // the chunks' sums take the place of dz and X
#pragma unroll
  for (int u = 0; u < KT; ++u)
    *reinterpret_cast<float4*>(&ds[(c * COLS + kq + u) * kHidden + jq]) = make_float4(s[u][0], s[u][1], s[u][2], s[u][3]);
  if (kq == 0) *reinterpret_cast<float4*>(&xs[c * kHidden + jq]) = make_float4(sb[0], sb[1], sb[2], sb[3]);
  __syncthreads();
#pragma unroll
  for (int o = threadIdx.x; o < COLS * kHidden; o += 256) {
    double acc = 0.0;
#pragma unroll
    for (int h = 0; h < NCH; ++h) acc += (double)ds[h * COLS * kHidden + o];
    const int k = k0 + o / kHidden;
    if (k < KIN) part[(long)(k * kHidden + o % kHidden) * cap + blk] = acc;
  }
  if (k0 == 0 && threadIdx.x < kHidden) {
    double acc = 0.0;
#pragma unroll
    for (int h = 0; h < NCH; ++h) acc += (double)xs[h * kHidden + threadIdx.x];
    part[(long)(KIN * kHidden + threadIdx.x) * cap + blk] = acc;
  }
}
template <int KIN, int COLS>
void wgrad_partials(hipStream_t s, int n, const float* X0, int ld0, int c0, const float* X1, int ld1, int kin,
                    const float* dz, const float* Zm, double* part, int cap) {
  static_assert(COLS % 4 == 0 && COLS <= 32, "the chunks' sums fit where dz was");
  const long g = (cap + kXcds - 1) / kXcds * kXcds * ((KIN + COLS - 1) / COLS);
  hipLaunchKernelGGL((k_wgrad_partials<KIN, COLS>), dim3((unsigned)g), dim3(256), 0, s, n, X0, ld0, c0, X1, ld1, kin,
                     dz, Zm, part, cap);
}

// out[o] (+)= sum_b part[o * cap + b] in block order. A workgroup takes kColOut outputs: tiles of 256 partials of
// each are loaded coalesced, the next while one lane per output adds the last, so that a tile costs its chain of
// additions (one lane per output reading 8 bytes of a line at a time took 449 us at 96^3, this 71; at 16^3 both 3.4).
constexpr int kColOut = 8;
__global__ void __launch_bounds__(256) k_colsum(int nout, int nblk, const double* __restrict__ part, int cap,
                                                float* __restrict__ out, int accumulate) {
  __shared__ double tile[kColOut][256 + 1];
  const int o0 = blockIdx.x * kColOut, t = threadIdx.x;
  double v[kColOut], s = 0.0;
  auto load = [&](int b0) {
#pragma unroll
    for (int c = 0; c < kColOut; ++c)
      v[c] = o0 + c < nout && b0 + t < nblk ? part[(long)(o0 + c) * cap + b0 + t] : 0.0;
  };
  load(0);
  for (int b0 = 0; b0 < nblk; b0 += 256) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < kColOut; ++c) tile[c][t] = v[c];
    __syncthreads();
    load(b0 + 256);
    if (t < kColOut) {
      const int m = min(256, nblk - b0);
#pragma unroll 16
      for (int b = 0; b < m; ++b) s += tile[t][b];
    }
  }
  const int o = o0 + t;
  if (t < kColOut && o < nout) out[o] = accumulate ? out[o] + (float)s : (float)s;
}
// per-row head gradient terms (N x kHeadGrads) -> partials per 256 rows. A workgroup takes kRowsumCols of the
// columns through LDS (every load in flight at once); one lane then adds a column's rows in order.
// Lanes that walked their column in memory had few loads in flight: 41 us at 16^3, now 5.5.
constexpr int kRowsumCols = 25;
__global__ void __launch_bounds__(256) k_rowsum_partials(int n, int ncol, const float* __restrict__ prow,
                                                         double* __restrict__ part, int cap) {
  __shared__ float xs[256 * kRowsumCols];
  const int r0 = blockIdx.x * 256, o0 = blockIdx.y * kRowsumCols, rows = min(256, n - r0);
  float v[kRowsumCols];
#pragma unroll
  for (int q = 0; q < kRowsumCols; ++q) {
    const int t = q * 256 + threadIdx.x, r = t / kRowsumCols, o = o0 + t % kRowsumCols;
    v[q] = r < rows && o < ncol ? prow[(long)(r0 + r) * ncol + o] : 0.f;
  }
#pragma unroll
  for (int q = 0; q < kRowsumCols; ++q) xs[q * 256 + threadIdx.x] = v[q];
  __syncthreads();
  const int o = o0 + threadIdx.x;
  if (threadIdx.x >= kRowsumCols || o >= ncol) return;
  double s = 0.0;
#pragma unroll 16
  for (int r = 0; r < rows; ++r) s += (double)xs[r * kRowsumCols + threadIdx.x];
  part[(long)o * cap + blockIdx.x] = s;
}

// Adam (Kingma & Ba 2015) on the FP32 master weights
__global__ void k_adam(int np, float* __restrict__ P, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  P[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Transpose positions: tpos[k] = position of (j, i) in row j for the entry
// k = (i, j); a missing mirror entry (pattern not symmetric) raises *bad.
__global__ void k_tpos(int n, const int* __restrict__ ro, const int* __restrict__ cols, const int* __restrict__ dcol,
                       const double* __restrict__ vals, int* __restrict__ tpos, int* __restrict__ bad) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int d = dcol[i];
  if (d >= ro[i + 1] || cols[d] != i) atomicOr(bad, 2);
  else if (!(vals[d] > 0)) atomicOr(bad, 4);
  for (int k = ro[i]; k < ro[i + 1]; ++k) {
    const int j = cols[k];
    int q = -1;
    for (int t = ro[j]; t < ro[j + 1]; ++t)
      if (cols[t] == i) {
        q = t;
        break;
      }
    tpos[k] = q;
    if (q < 0) atomicOr(bad, 1);
  }
}

// a factor value in its storage type: FP64, FP32, or bfloat16 (FP32 rounded to
// nearest even, then its upper half rounded to nearest even)
template <typename T>
__device__ __forceinline__ T factor_store(double g) {
  return (T)g;
}
template <>
__device__ __forceinline__ bf16_bits factor_store<bf16_bits>(double g) {
  return (bf16_bits)to_bf16((float)g);
}

// Row-bundled values of G (TRANS = false: rows = lower + diagonal of A,
// G_ij = dis_i Ghat_ij) or of G^T (TRANS: rows = diagonal + upper, (G^T)_ij =
// G_ji = dis_j Ghat_ji, read at the transpose position). Lane = row; the row's
// entries are walked together with the bundle's slots: slot j of an RB-CSR
// bundle is the row's j-th entry, an RB-DIA slot the entry at offset doff.
template <typename T, bool TRANS>
__global__ void k_fill_factor(int n, const int* __restrict__ ro, const int* __restrict__ cols,
                              const int* __restrict__ dcol, const int* __restrict__ tpos, const int* __restrict__ bo,
                              const int* __restrict__ doff, const float* __restrict__ ghat,
                              const float* __restrict__ dis, T* __restrict__ bv) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int nb = (n + kBundle - 1) / kBundle;
  const int b = t / kBundle, lane = t % kBundle;
  if (b >= nb) return;
  const int row = t;
  const int s0 = bo[b], w = bo[b + 1] - s0;
  int k = 0, e = 0;
  if (row < n) {
    k = TRANS ? dcol[row] : ro[row];
    e = TRANS ? ro[row + 1] : dcol[row] + 1;
  }
  for (int j = 0; j < w; ++j) {
    T v = T(0);
    if (k < e && (!doff || cols[k] - row == doff[s0 + j])) {
      const double g = TRANS ? (double)dis[cols[k]] * (double)ghat[tpos[k]] : (double)dis[row] * (double)ghat[k];
      v = factor_store<T>(g);
      ++k;
    }
    bv[((long)s0 + j) * kBundle + lane] = v;
  }
}

} // namespace gnn
} // namespace alien_hip

// =====================================================================================
// Host engine: device buffers of one system and the launch sequences
// =====================================================================================
#include "../alien/hip/HIPContext.h"

namespace alien_hip {
namespace gnn {

namespace {
inline dim3 g1(long n, int b = 256) { return dim3((unsigned)((n + b - 1) / b)); }
} // namespace

Engine::Engine(alien_hip_ctx* ctx, int n, const int* ro, const int* cols, const double* vals) : m_ctx(ctx), m_n(n) {
  const int nnz = ro[n];
  h_ro.assign(ro, ro + n + 1);
  h_cols.assign(cols, cols + nnz);
  h_dcol.resize(n);
  host_dcol(n, ro, cols, h_dcol.data());
  hipStream_t s = m_ctx->stream;
  d_ro.upload(h_ro.data(), h_ro.size(), s);
  d_cols.upload(h_cols.data(), h_cols.size(), s);
  d_dcol.upload(h_dcol.data(), h_dcol.size(), s);
  d_vals.upload(vals, nnz, s);
  SystemView v;
  v.n = n;
  v.ro = h_ro.data();
  v.cols = h_cols.data();
  v.dcol = h_dcol.data();
  v.vals = vals;
  v.d_ro = d_ro.data();
  v.d_cols = d_cols.data();
  v.d_dcol = d_dcol.data();
  v.d_vals = d_vals.data();
  init(v);
}

Engine::Engine(alien_hip_ctx* ctx, const SystemView& v) : m_ctx(ctx), m_n(v.n) { init(v); }

// Checks of the system (stored positive diagonal, symmetric pattern), the
// transpose positions and the per-system buffers; host values are read here only.
void Engine::init(const SystemView& v) {
  const int n = v.n;
  m_nnz = v.ro[n];
  m_v = v;
  m_v.vals = nullptr;
  hipStream_t s = m_ctx->stream;
  d_tpos.resize(m_nnz);
  {
    // transpose positions, and the checks of the stored diagonal and the pattern's symmetry
    DeviceArray<int> bad(1);
    ALIEN_HIP_CHECK(hipMemsetAsync(bad.data(), 0, sizeof(int), s));
    hipLaunchKernelGGL(k_tpos, g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol, m_v.d_vals, d_tpos.data(),
                       bad.data());
    check_launch("gnn tpos");
    int hbad = 0;
    ALIEN_HIP_CHECK(hipMemcpyAsync(&hbad, bad.data(), sizeof(int), hipMemcpyDeviceToHost, s));
    ALIEN_HIP_CHECK(hipStreamSynchronize(s));
    if (hbad & 2) throw Error(ALIEN_HIP_EINVAL, "learned preconditioner: missing diagonal");
    if (hbad & 4) throw Error(ALIEN_HIP_EINVAL, "learned preconditioner: non-positive diagonal");
    if (hbad & 1) throw Error(ALIEN_HIP_EINVAL, "learned preconditioner: the pattern must be symmetric");
  }
  d_dis.resize(n);
  d_e.resize(m_nnz);
  d_f.resize((size_t)n * kFeat);
  d_ghat.resize(m_nnz);
}

// Activation buffers (n x 32 each): every layer's input, pre-activation and
// message for the backward pass, or two inputs and one message for inference.
void Engine::ensure_activations(bool all_layers) {
  const size_t sz = (size_t)m_n * kHidden;
  for (int l = 0; l < 4; ++l) {
    const bool need_h = all_layers || l < 2, need_z = all_layers, need_m = all_layers || l == 1;
    if (need_h && d_h[l].empty()) d_h[l].resize(sz);
    if (need_z && d_z[l].empty()) d_z[l].resize(sz);
    if (need_m && d_m[l].empty()) d_m[l].resize(sz);
  }
}

// scaled couplings and node features from A's values
void Engine::prep_features() {
  hipStream_t s = m_ctx->stream;
  const int n = m_n;
  hipLaunchKernelGGL(k_prep_dis, g1(n), dim3(256), 0, s, n, m_v.d_dcol, m_v.d_vals, d_dis.data());
  hipLaunchKernelGGL(k_prep_feat, g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_vals, d_dis.data(),
                     d_e.data(), d_f.data());
}

void Engine::forward(const float* P) {
  ensure_activations(true);
  hipStream_t s = m_ctx->stream;
  const int n = m_n;
  prep_features();
  const dim3 gd((unsigned)(((n + 31) / 32 + 3) / 4)); // 32 rows per wavefront, 4 wavefronts per workgroup
  hipLaunchKernelGGL(k_dense<8>, gd, dim3(256), 0, s, n, d_f.data(), kFeat, kFeat, (const float*)nullptr, 0, kFeat,
                     P + kOffWin, P + kOffBin, (const float*)nullptr, d_z[0].data(), d_h[0].data());
  const int offs[3] = {kOffW1, kOffW2, kOffW3};
  for (int l = 1; l <= 3; ++l) {
    hipLaunchKernelGGL(k_aggregate, aggregate_grid(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, d_e.data(),
                       d_h[l - 1].data(), d_m[l].data());
    hipLaunchKernelGGL(k_dense<64>, gd, dim3(256), 0, s, n, d_h[l - 1].data(), kHidden, kHidden, d_m[l].data(), kHidden,
                       2 * kHidden, P + offs[l - 1], P + offs[l - 1] + 2 * kHidden * kHidden, d_h[l - 1].data(),
                       d_z[l].data(), d_h[l].data());
  }
  hipLaunchKernelGGL(k_head, g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol, d_e.data(),
                     d_h[3].data(), P, d_ghat.data());
  check_launch("gnn forward");
}

// The same arithmetic as forward(), layer l reading buffer (l - 1) % 2 and
// writing l % 2, pre-activations not stored.
void Engine::infer(const float* P) {
  ensure_activations(false);
  hipStream_t s = m_ctx->stream;
  const int n = m_n;
  prep_features();
  const dim3 gd((unsigned)(((n + 31) / 32 + 3) / 4));
  hipLaunchKernelGGL(k_dense<8>, gd, dim3(256), 0, s, n, d_f.data(), kFeat, kFeat, (const float*)nullptr, 0, kFeat,
                     P + kOffWin, P + kOffBin, (const float*)nullptr, (float*)nullptr, d_h[0].data());
  const int offs[3] = {kOffW1, kOffW2, kOffW3};
  for (int l = 1; l <= 3; ++l) {
    const float* hin = d_h[(l - 1) & 1].data();
    float* hout = d_h[l & 1].data();
    hipLaunchKernelGGL(k_aggregate, aggregate_grid(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, d_e.data(), hin,
                       d_m[1].data());
    hipLaunchKernelGGL(k_dense<64>, gd, dim3(256), 0, s, n, hin, kHidden, kHidden, d_m[1].data(), kHidden,
                       2 * kHidden, P + offs[l - 1], P + offs[l - 1] + 2 * kHidden * kHidden, hin, (float*)nullptr,
                       hout);
  }
  hipLaunchKernelGGL(k_head, g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol, d_e.data(),
                     d_h[1].data(), P, d_ghat.data());
  check_launch("gnn inference");
}

double Engine::loss_grad(const float* P, const float* V, int K, float beta, int cg_steps, float* grad,
                         double* parts) {
  if (K != 4) throw Error(ALIEN_HIP_EINVAL, "learned preconditioner: 4 probe vectors are supported");
  if (cg_steps < 0 || cg_steps > kMaxCgSteps) throw Error(ALIEN_HIP_EINVAL, "learned preconditioner: bad cg_steps");
  hipStream_t s = m_ctx->stream;
  const int n = m_n;
  forward(P);
  // ---- Kaporin term (cg_steps == 0)
  m_ctx->reserve_for(n);
  DeviceArray<float> ag(m_nnz), gg(m_nnz);
  DeviceArray<double> sums(4);
  const long nb = (n + 255) / 256;
  RedWork w = m_ctx->red();
  const bool kap = cg_steps == 0;
  if (kap) {
    hipLaunchKernelGGL(k_kcond, dim3((unsigned)nb), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol,
                       d_tpos.data(), d_e.data(), d_ghat.data(), ag.data(), w);
    launch_finalize(s, w, nb, 2, kFinStore, sums.data(), nullptr);
  }
  // ---- probe term
  constexpr int KP = 4;
  DeviceArray<float> W_((size_t)n * KP), U((size_t)n * KP), Y((size_t)n * KP), dY((size_t)n * KP), Q((size_t)n * KP);
  hipLaunchKernelGGL((k_ahat_mult<KP>), g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, d_e.data(), V, W_.data());
  hipLaunchKernelGGL((k_ghat_mult<KP, true>), g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol,
                     d_tpos.data(), d_ghat.data(), W_.data(), U.data());
  hipLaunchKernelGGL((k_ghat_mult<KP, false>), g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol,
                     d_tpos.data(), d_ghat.data(), U.data(), Y.data());
  hipLaunchKernelGGL((k_probe_resid<KP>), dim3((unsigned)nb), dim3(256), 0, s, n, V, Y.data(), dY.data(),
                     (float)(1.0 / ((double)n * KP)), w);
  launch_finalize(s, w, nb, 1, kFinStore, sums.data() + 2, nullptr);
  hipLaunchKernelGGL((k_ghat_mult<KP, true>), g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol,
                     d_tpos.data(), d_ghat.data(), dY.data(), Q.data());
  hipLaunchKernelGGL((k_grad_ghat<KP>), g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol,
                     d_ghat.data(), ag.data(), sums.data(), kap ? 1.f : 0.f, beta, dY.data(), U.data(), W_.data(),
                     Q.data(), gg.data());
  // ---- CG term (cg_steps > 0): k PCG steps on Ahat with Ghat Ghat^T, reverse pass into gg
  double lcg = 0.0;
  if (!kap) lcg = cg_term(V, cg_steps, gg.data());
  // ---- head backward
  DeviceArray<float> dh[2], dz((size_t)n * kHidden), dmsg((size_t)n * kHidden), prow((size_t)n * kHeadGrads);
  dh[0].resize((size_t)n * kHidden);
  dh[1].resize((size_t)n * kHidden);
  hipLaunchKernelGGL(k_head_bwd, g1(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols, m_v.d_dcol, d_tpos.data(),
                     d_e.data(), d_ghat.data(), gg.data(), d_h[3].data(), P, dh[0].data(), prow.data());
  const int cap = (int)nb;
  DeviceArray<double> part((size_t)(2 * kHidden * kHidden + kHidden) * cap);
  hipLaunchKernelGGL(k_rowsum_partials, dim3((unsigned)nb, (kHeadGrads + kRowsumCols - 1) / kRowsumCols), dim3(256), 0, s, n, kHeadGrads, prow.data(), part.data(), cap);
  hipLaunchKernelGGL(k_colsum, g1(kHeadGrads, kColOut), dim3(256), 0, s, kHeadGrads, (int)nb, part.data(), cap, grad + kOffWd, 0);
  // ---- message-passing layers, last to first
  const int offs[3] = {kOffW1, kOffW2, kOffW3};
  int cur = 0;
  for (int l = 3; l >= 1; --l) {
    const float* Wl = P + offs[l - 1];
    hipLaunchKernelGGL(k_dense_bwd_mfma, dim3((unsigned)(((n + 31) / 32 + 3) / 4)), dim3(256), 0, s, n, dh[cur].data(),
                       d_z[l].data(), Wl, dz.data(), dh[cur ^ 1].data(), dmsg.data());
    hipLaunchKernelGGL(k_aggregate_add, aggregate_grid(n), dim3(256), 0, s, n, m_v.d_ro, m_v.d_cols,
                       d_tpos.data(), d_e.data(), dmsg.data(), dh[cur ^ 1].data());
    if (nb < kWgradWide)
      wgrad_partials<2 * kHidden, 8>(s, n, d_h[l - 1].data(), kHidden, kHidden, d_m[l].data(), kHidden, 2 * kHidden,
                                     dz.data(), nullptr, part.data(), cap);
    else
      wgrad_partials<2 * kHidden, 32>(s, n, d_h[l - 1].data(), kHidden, kHidden, d_m[l].data(), kHidden, 2 * kHidden,
                                      dz.data(), nullptr, part.data(), cap);
    hipLaunchKernelGGL(k_colsum, g1(kLayerSize, kColOut), dim3(256), 0, s, kLayerSize, (int)nb, part.data(), cap,
                       grad + offs[l - 1], 0);
    cur ^= 1;
  }
  // ---- input layer
  wgrad_partials<kFeat, 8>(s, n, d_f.data(), kFeat, kFeat, nullptr, 0, kFeat, dh[cur].data(), d_z[0].data(),
                           part.data(), cap);
  hipLaunchKernelGGL(k_colsum, g1(kFeat * kHidden + kHidden, kColOut), dim3(256), 0, s, kFeat * kHidden + kHidden, (int)nb,
                     part.data(), cap, grad + kOffWin, 0);
  check_launch("gnn backward");
  double hs[4];
  ALIEN_HIP_CHECK(hipMemcpyAsync(hs, sums.data(), 3 * sizeof(double), hipMemcpyDeviceToHost, s));
  ALIEN_HIP_CHECK(hipStreamSynchronize(s));
  const double lk = kap ? std::log(hs[0] / n) - 2.0 * hs[1] / n : lcg;
  const double lp = hs[2] / ((double)n * KP);
  if (parts) {
    parts[0] = lk;
    parts[1] = lp;
  }
  return lk + beta * lp;
}

// Residual reduction after k PCG steps on Ahat with M = Ghat Ghat^T, x0 = 0, the
// 4 columns of B as right-hand sides: L = mean_c log(|r_k|^2 / |r_0|^2), rho =
// |Ghat^T r|^2. Forward keeps r_j, t_j = Ghat^T r_j, p_j, q_j = Ahat p_j; the
// reverse pass (the adjoint of each step, last to first) accumulates dL/dGhat
// on the lower pattern into gg. Three launches a step each way; the host reads
// |r_0|^2 and |r_k|^2 once, between the two. Vectors in FP32, dots in FP64.
double Engine::cg_term(const float* B, int k, float* gg) {
  hipStream_t s = m_ctx->stream;
  const int n = m_n;
  const long nb = (n + 255) / 256;
  const dim3 g((unsigned)nb), t256(256);
  // vectors: r_0..r_k, t_j, p_j, q_j (j < k) and the adjoints of r, p and t
  DeviceArray<float4> vec((size_t)n * (4 * (size_t)k + 4));
  auto at = [&](size_t slot) { return vec.data() + slot * (size_t)n; };
  auto R = [&](int j) { return at(j); };
  auto T = [&](int j) { return at((size_t)k + 1 + j); };
  auto Pv = [&](int j) { return at(2 * (size_t)k + 1 + j); };
  auto Q = [&](int j) { return at(3 * (size_t)k + 1 + j); };
  float4 *rbar = at(4 * (size_t)k + 1), *pbar = at(4 * (size_t)k + 2), *tbar = at(4 * (size_t)k + 3);
  // partials of two dot products in turn (a kernel consumes one and produces the next) and of r_0.r_0,
  // a total, and the step scalars kept on the device
  DeviceArray<double> dots(12 * (size_t)nb + 12 + 16 * (size_t)k);
  double* part[2] = {dots.data(), dots.data() + 4 * nb};
  double* rr_part = dots.data() + 8 * nb;
  double* tot = dots.data() + 12 * nb;
  double *rr = tot + 4, *scal = tot + 12;
  auto rho = [&](int j) { return scal + 4 * (size_t)j; };
  auto sig = [&](int j) { return scal + 4 * (size_t)(k + j); };
  auto own = [&](int j) { return scal + 4 * (size_t)(2 * k + j); };
  auto rhobar = [&](int j) { return scal + 4 * (size_t)(3 * k + j); };
  int cur = 0; // part[cur] holds the last dot product's partials
  auto next = [&] { return part[cur ^= 1]; };
  // Up to a wavefront's lanes of partials are summed by their consumers; more take the finalize's launch
  // (4.5 us), which costs less than every wavefront of the consumer reading several rounds of them.
  auto value = [&]() {
    if (nb <= kWave) return Dot4{part[cur], (int)nb};
    launch_finalize(s, RedWork{part[cur], (int)nb}, nb, 4, kFinStore, tot, nullptr);
    return Dot4{tot, 1};
  };
  const CgRows A{n, m_v.d_ro, m_v.d_cols, m_v.d_dcol, d_tpos.data(), d_e.data(), d_ghat.data()};
  // forward
  ALIEN_HIP_CHECK(hipMemcpyAsync(R(0), B, sizeof(float4) * n, hipMemcpyDeviceToDevice, s));
  hipLaunchKernelGGL(k_cg4_start, g, t256, 0, s, A, R(0), T(0), next(), rr_part, (int)nb);
  for (int j = 0; j < k; ++j) {
    const Dot4 rho1 = value();
    hipLaunchKernelGGL(k_cg4_dir, g, t256, 0, s, A, T(j), j ? Pv(j - 1) : (const float4*)nullptr, rho1,
                       j ? rho(j - 1) : (const double*)nullptr, rho(j), Pv(j));
    hipLaunchKernelGGL(k_cg4_ap, g, t256, 0, s, A, Pv(j), Q(j), next(), (int)nb);
    const Dot4 pq = value();
    hipLaunchKernelGGL(k_cg4_res, g, t256, 0, s, A, R(j), Q(j), rho(j), pq, sig(j), R(j + 1),
                       j < k - 1 ? T(j + 1) : (float4*)nullptr, next(), (int)nb);
  }
  launch_finalize(s, RedWork{rr_part, (int)nb}, nb, 4, kFinStore, rr, nullptr);
  launch_finalize(s, RedWork{part[cur], (int)nb}, nb, 4, kFinStore, rr + 4, nullptr);
  check_launch("gnn cg loss");
  double h[8]; // |r_0|^2, |r_k|^2
  m_ctx->read_words(rr, h, 16);
  double L = 0.0;
  Coef4 c0;
  for (int c = 0; c < 4; ++c) {
    L += std::log(h[4 + c] / h[c]) / 4.0;
    c0.c[c] = (float)(2.0 / (4.0 * h[4 + c]));
  }
  if (!std::isfinite(L)) return L;
  // reverse
  hipLaunchKernelGGL(k_cg4_rev_start, g, t256, 0, s, n, c0, R(k), Q(k - 1), rbar, next(), (int)nb);
  for (int j = k - 1; j >= 0; --j) {
    const bool last = j == k - 1; // p_k is not formed
    if (!last) {
      const Dot4 betabar = value();
      hipLaunchKernelGGL(k_cg4_rev_t, g, t256, 0, s, A, pbar, T(j + 1), rhobar(j + 1), betabar, rho(j), rho(j + 1),
                         own(j), tbar);
      hipLaunchKernelGGL(k_cg4_rev_r, g, t256, 0, s, A, pbar, T(j + 1), R(j + 1), tbar, gg, rbar, Q(j), next(),
                         (int)nb);
    }
    const Dot4 qr = value();
    hipLaunchKernelGGL(k_cg4_rev_p, g, t256, 0, s, A, rbar, Pv(j), Q(j), rho(j),
                       last ? (const double*)nullptr : rho(j + 1), sig(j), qr, own(j), rhobar(j), pbar,
                       j ? Pv(j - 1) : (const float4*)nullptr, next(), (int)nb);
  }
  // p_0 = Ghat t_0, rho_0 = t_0.t_0, t_0 = Ghat^T r_0
  hipLaunchKernelGGL(k_cg4_rev_t, g, t256, 0, s, A, pbar, T(0), rhobar(0), Dot4{nullptr, 0}, (const double*)nullptr,
                     (const double*)nullptr, (double*)nullptr, tbar);
  hipLaunchKernelGGL(k_cg4_rev_r, g, t256, 0, s, A, pbar, T(0), R(0), tbar, gg, (float4*)nullptr,
                     (const float4*)nullptr, (double*)nullptr, (int)nb);
  check_launch("gnn cg loss");
  ALIEN_HIP_CHECK(hipStreamSynchronize(s)); // before the vectors are freed
  return L;
}

// Row-bundled layouts of G (rows = lower + diagonal of A) and of G^T (rows =
// diagonal + upper of A; the pattern is symmetric): RB-DIA when it stores at
// most kRbdiaMaxGrowth times the RB-CSR slots, RB-CSR otherwise. When A itself
// is RB-DIA, the factors' offsets and lane masks are A's with offset <= 0 (G)
// and >= 0 (G^T): a split of A's structure, no pass over the entries.
void Engine::build_factor_layout() {
  if (!m_gbo.empty()) return;
  const int n = m_n;
  const int nb = (n + kBundle - 1) / kBundle;
  hipStream_t s = m_ctx->stream;
  const bool split = m_v.rb_bo && m_v.d_rb_doff && m_v.d_rb_dmask;
  std::vector<int> adoff;
  std::vector<unsigned long long> admask;
  if (split) {
    const size_t aslots = (size_t)m_v.rb_bo[nb];
    adoff.resize(aslots);
    admask.resize(aslots);
    ALIEN_HIP_CHECK(hipMemcpyAsync(adoff.data(), m_v.d_rb_doff, aslots * sizeof(int), hipMemcpyDeviceToHost, s));
    ALIEN_HIP_CHECK(hipMemcpyAsync(admask.data(), m_v.d_rb_dmask, aslots * sizeof(unsigned long long),
                                   hipMemcpyDeviceToHost, s));
    ALIEN_HIP_CHECK(hipStreamSynchronize(s));
  }
  // RB-CSR widths of both factors in one pass: row r of G has dcol - ro + 1 entries, of G^T ro' - dcol
  std::vector<int> cbos[2] = {std::vector<int>(nb + 1, 0), std::vector<int>(nb + 1, 0)};
  long totals[2] = {0, 0};
  {
    long* acc = totals;
    for (int b = 0; b < nb; ++b) {
      cbos[0][b] = (int)acc[0];
      cbos[1][b] = (int)acc[1];
      int w0 = 0, w1 = 0;
      for (int r = b * kBundle; r < std::min(n, (b + 1) * kBundle); ++r) {
        w0 = std::max(w0, m_v.dcol[r] - m_v.ro[r] + 1);
        w1 = std::max(w1, m_v.ro[r + 1] - m_v.dcol[r]);
      }
      acc[0] += w0;
      acc[1] += w1;
    }
    cbos[0][nb] = (int)acc[0];
    cbos[1][nb] = (int)acc[1];
  }
  std::vector<int> kb, ke; // entry ranges per row, built only for a host structure pass
  for (int t = 0; t < 2; ++t) {
    const std::vector<int>& cbo = cbos[t];
    const long acc = totals[t];
    auto ranges = [&]() {
      kb.resize(n);
      ke.resize(n);
      for (int r = 0; r < n; ++r) {
        kb[r] = t == 0 ? m_v.ro[r] : m_v.dcol[r];
        ke[r] = t == 0 ? m_v.dcol[r] + 1 : m_v.ro[r + 1];
      }
    };
    if (acc * kBundle > 0x7fffffffL) throw Error(ALIEN_HIP_EINVAL, "learned preconditioner: factor too large");
    std::vector<int> dbo, doff;
    std::vector<uint64_t> dmask;
    long dslots;
    if (split) {
      dbo.assign(nb + 1, 0);
      doff.reserve(adoff.size());
      dmask.reserve(adoff.size());
      for (int b = 0; b < nb; ++b) {
        dbo[b] = (int)doff.size();
        for (int j = m_v.rb_bo[b]; j < m_v.rb_bo[b + 1]; ++j) {
          if (t == 0 ? adoff[j] > 0 : adoff[j] < 0) continue;
          doff.push_back(adoff[j]);
          dmask.push_back(admask[j]);
        }
      }
      dbo[nb] = (int)doff.size();
      dslots = dbo[nb];
    } else {
      ranges();
      dslots = rbdia_structure(n, m_v.ro, m_v.cols, kb.data(), ke.data(), kRbdiaMaxWidth, dbo, doff, dmask);
    }
    const bool dia = dslots >= 0 && dslots <= kRbdiaMaxGrowth * cbo[nb];
    std::vector<int>& bo = t == 0 ? m_gbo : m_gtbo;
    bo = dia ? dbo : cbo;
    const size_t slots = (size_t)bo[nb] * kBundle;
    Factor& F = t == 0 ? m_g : m_gt;
    F.dia = dia;
    F.uni = 0;
    if (dia && nb > 0) {
      // uniform when every bundle holds the same offsets (the split of a uniform A)
      const int k = bo[1] - bo[0];
      bool same = k >= 1 && k <= kUniMaxSlots;
      for (int b = 0; same && b < nb; ++b) {
        same = bo[b] == b * k && bo[b + 1] == (b + 1) * k;
        for (int j = 0; same && j < k; ++j) same = doff[(size_t)b * k + j] == doff[j];
      }
      if (same) {
        F.uni = k;
        F.nrows = n;
        for (int j = 0; j < k; ++j) F.uoff[j] = doff[j];
      }
    }
    F.bo.upload(bo.data(), bo.size(), s);
    if (dia) {
      F.doff.upload(doff.data(), doff.size(), s);
      F.dmask.upload(reinterpret_cast<const unsigned long long*>(dmask.data()), dmask.size(), s);
    } else {
      ranges();
      std::vector<int> bc(slots, -1);
      for (int r = 0; r < n; ++r) {
        const int b = r / kBundle, lane = r % kBundle;
        for (int k = kb[r]; k < ke[r]; ++k) bc[((size_t)bo[b] + (k - kb[r])) * kBundle + lane] = m_v.cols[k];
      }
      F.bc.upload(bc.data(), slots, s);
    }
    F.slots = slots;
  }
  ALIEN_HIP_CHECK(hipStreamSynchronize(s));
}

template <typename T>
void Engine::fill_factor(T* g_vals, T* gt_vals) {
  build_factor_layout();
  hipStream_t s = m_ctx->stream;
  const int nrows64 = (m_n + kBundle - 1) / kBundle * kBundle;
  hipLaunchKernelGGL((k_fill_factor<T, false>), g1(nrows64), dim3(256), 0, s, m_n, m_v.d_ro, m_v.d_cols,
                     m_v.d_dcol, d_tpos.data(), m_g.bo.data(), m_g.dia ? m_g.doff.data() : nullptr,
                     d_ghat.data(), d_dis.data(), g_vals);
  hipLaunchKernelGGL((k_fill_factor<T, true>), g1(nrows64), dim3(256), 0, s, m_n, m_v.d_ro, m_v.d_cols,
                     m_v.d_dcol, d_tpos.data(), m_gt.bo.data(), m_gt.dia ? m_gt.doff.data() : nullptr,
                     d_ghat.data(), d_dis.data(), gt_vals);
  check_launch("gnn fill factor");
}
void Engine::release_network_buffers() {
  ALIEN_HIP_CHECK(hipStreamSynchronize(m_ctx->stream));
  for (int l = 0; l < 4; ++l) {
    d_h[l].reset();
    d_z[l].reset();
    d_m[l].reset();
  }
  d_e.reset();
  d_f.reset();
  d_ghat.reset();
  d_dis.reset();
  d_tpos.reset();
}

template void Engine::fill_factor<float>(float*, float*);
template void Engine::fill_factor<bf16_bits>(bf16_bits*, bf16_bits*);
template void Engine::fill_factor<double>(double*, double*);

void launch_adam(hipStream_t s, int np, float* P, const float* g, float* m, float* v, float lr, int step) {
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = 1.f - std::pow(b1, (float)step), c2 = 1.f - std::pow(b2, (float)step);
  hipLaunchKernelGGL(k_adam, g1(np), dim3(256), 0, s, np, P, g, m, v, lr, b1, b2, 1e-8f, c1, c2);
}

} // namespace gnn
} // namespace alien_hip
