// CG iterations of small and middle-sized systems in one launch, the system held in registers.
//
// An iteration of the fused CG is five to nine dependent launches (krylov.hip), each 3.5-4.8 us
// however small the system: 20-40 us an iteration below a few hundred thousand rows, where the
// memory traffic would take one or two. Here one launch holds 1024 R rows per compute unit, R rows
// per lane: their matrix entries, x, r, the inverse diagonal and the search direction at the rows'
// own columns stay in registers, and an iteration costs two grid-wide sums (p.q; r.r and r.z) and
// one exchange of z. p is not exchanged: a lane updates its copies p[c] = z[c] + beta p[c] by the
// owner's operation on the owner's operands, so they are the owner's values. The Chebyshev
// preconditioner adds a sum and an exchange per step.
// Element-wise operations are those of krylov.hip in the same order, and the sums follow the same
// trees (lanes, wavefronts, workgroups and finalize of the launches), so the iterates are the
// launches' bit for bit.
// Every workgroup has to be running: there are no more than compute units, a workgroup fits beside
// any other kernel's once that ends, and the caller lets such launches of the process run together only where
// the compute units hold them all (ResidentTurn); what else might hold one back too long runs the waits out of polls.
// Bound by the latency of the sums, about 3 us each, and in one workgroup by its instructions. An iteration of
// Jacobi-CG in FP64 against the graph of launches: 14 x 11 x 9 cells 2.8 us (16), 32^3 5.6 (18), 64^3 8.5 (21), 80^3 (two
// rows per lane, which spill) 22 (30); FP32 in the mixed solver 7.9 (19) at 64^3; Chebyshev of degree 3 16 (39) at
// 32^3. Each barrier of a sum costs some 0.1 us: one after the totals are read was spared by a place of their own
// (64^3 mixed 9.1 -> 8.7 us a solve's iteration), two sets of places in turn, indexed, cost more than they spared (10.3).
// One sum per workgroup, with a tree of its own, took 7.7 us at 64^3, but its iterates are not the launches'.
// Exchanging through barriers (stores settled, then a sum, then loads) took 10.4.
#include "../alien_hip_internal.h"
#include "../alien/hip/HIPContext.h"
#include "device_common.h"
#include "krylov_state.h"
#include "launch.h"
#include "rb_rows.h"
#include "sync_free.h"
#include "wave_total.h"

#include <type_traits>

namespace alien_hip {


template <typename T>
__device__ __forceinline__ T agent_load(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void agent_store(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Grid-wide sums over a launch of at most one workgroup per compute unit, as the launches take them.
// The rows' terms become the partials of the launches' workgroups, by KIND:
//   kSumRows   row kernels, a wavefront per bundle: partial l of rows 256 l .. (krylov.hip)
//   kSumPairs  the uniform layout's q = A p, a wavefront per two bundles: partial l of rows 512 l ..
//   kSumStream streaming kernels, kEPT elements 256 apart per lane: partial l of elements 1024 l ..
// the first two under the workgroup number that bundle_walk gives them. Partials are published as two
// words, half of their bits and the phase number in either, and every workgroup reads all of them
// until their phase is this one: no counter, nothing to clear, and a word is never taken from
// another phase. Two sets of slots are used in turn: a workgroup writes a set again only after a
// phase that every workgroup reached by having read it. Then each adds them as k_finalize does.
// settle: the agent-scope stores made before the call by any lane are complete at that scope when a
// workgroup returns from it anywhere (each wavefront waits for its own first).
// false: a wait ran out of polls, here or (failed) before.
constexpr int kResBlock = 1024; // lanes of a workgroup, as of k_finalize; R rows of a lane are 1024 apart
constexpr int kResWaves = kResBlock / kWave;
enum SumKind { kSumRows = 0, kSumPairs = 1, kSumStream = 2 };
struct GridSums {
  unsigned long long* slots;
  int* head; // [0] last phase, [1] a wait ran out of polls
  unsigned phase;
  long limit;
};
__device__ __forceinline__ bool give_up(const GridSums& g, long spins, int* failed) {
  if (spins <= g.limit && ((spins & 255) != 0 || !agent_load(g.head + 1))) return false;
  agent_store(g.head + 1, 1);
  *failed = 1;
  return true;
}
struct SumLds {
  double term[2][2][kResBlock]; // by value and round
  double wave[2][2][kResWaves], fin[2][kResWaves];
  double one[2][2][2][kResWaves]; // block_total's, by turn: none of its sums waits for the readers of the last
  int failed;
};
// The same within a launch of one workgroup. Its partials, at most 8, lie in the first 64 slots (bundle_walk
// gives row block l < 64 workgroup 8 l): after one or two barriers every wavefront adds them by the finalize's tree for
// itself.
template <int KIND, int NV, int R>
__device__ __forceinline__ void block_total(unsigned& phase, int n, const double (&term)[NV][R], double (&out)[NV], SumLds& L) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
  constexpr int W = kRowWaves, G = KIND == kSumRows ? 4 : KIND == kSumPairs ? 2 : 1;
  static_assert(G * R <= kWave / kXcds && (int)kXcdChunk >= G * R, "row block l is workgroup 8 l");
  auto& wave = L.one[++phase & 1];
  if constexpr (KIND == kSumRows) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double s = wave_total(term[0][q]);
      if (lane == 0) wave[0][q][wid] = s;
    }
  } else if constexpr (KIND == kSumPairs) {
    if (wid & 1)
#pragma unroll
      for (int q = 0; q < R; ++q) L.term[0][q][tid] = term[0][q];
    __syncthreads();
    if (!(wid & 1))
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const double s = wave_total(term[0][q] + L.term[0][q][tid + kWave]);
        if (lane == 0) wave[0][q][wid / 2] = s;
      }
  } else {
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int q = 0; q < R; ++q) L.term[v][q][tid] = term[v][q];
    __syncthreads();
    if (wid < W * NV * R) {
      const int v = wid / W % NV, q = wid / W / NV;
      const double* t = L.term[v][q] + tid % kBlock;
      const double s = wave_total(((t[0] + t[kBlock]) + t[2 * kBlock]) + t[3 * kBlock]);
      if (lane == 0) wave[v][q][wid % W] = s;
    }
  }
  __syncthreads();
  const int real = (n + kResBlock / G - 1) / (kResBlock / G);
  const int l = KIND == kSumStream ? lane : lane % kXcds ? real : lane / kXcds;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    double acc = 0;
    if (l < real) {
      double s = 0;
#pragma unroll
      for (int w = 0; w < W; ++w) s += wave[v][l / G][l % G * W + w];
      acc += s;
    }
    out[v] = 0.0 + wave_total(acc);
  }
}
template <int KIND, int NV, bool ONE, int R>
__device__ __forceinline__ bool grid_sum(GridSums& g, int n, const double (&term)[NV][R], double (&out)[NV], SumLds& L,
                                         bool settle) {
  if constexpr (ONE) {
    block_total<KIND, NV, R>(g.phase, n, term, out, L);
    return true;
  }
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid / kWave;
  constexpr int W = kRowWaves; // wavefronts of a launch's workgroup, whose totals are added in turn
  static_assert(R <= 2 && NV <= 2 && W * NV * R <= kResWaves, "");
  static_assert(kRowBlock == kBlock && kBlock * kEPT == kResBlock, "a workgroup holds whole workgroups of the launches");
  ++g.phase;
  if (settle) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  constexpr int G = KIND == kSumRows ? 4 : KIND == kSumPairs ? 2 : 1; // partials per 1024 rows
  const int per = kResBlock / G, real = (n + per - 1) / per;
  constexpr int C = (int)kXcdChunk, XC = kXcds * C;
  // slots of the launch's workgroups (`real` of them have rows), slot of workgroup l in row order, and back
  const int nslots = KIND == kSumStream ? real : ((n + kRowBlock - 1) / kRowBlock + XC - 1) / XC * XC;
  auto slot_of = [&](int l) { return KIND == kSumStream ? l : (l / XC * C + l % C) * kXcds + l / C % kXcds; };
  auto row_order = [&](int p) {
    const int i = p / kXcds;
    return KIND == kSumStream ? p : i / C * XC + p % kXcds * C + i % C;
  };
  unsigned long long* set = g.slots + (g.phase & 1) * (kResidentSlots * 4);
  const unsigned long long tag = (unsigned long long)g.phase << 32;
  if constexpr (KIND == kSumRows) {
#pragma unroll
    for (int q = 0; q < R; ++q) {
      const double s = wave_total(term[0][q]);
      if (lane == 0) L.wave[0][q][wid] = s;
    }
  } else if constexpr (KIND == kSumPairs) {
    if (wid & 1)
#pragma unroll
      for (int q = 0; q < R; ++q) L.term[0][q][tid] = term[0][q];
    __syncthreads();
    if (!(wid & 1))
#pragma unroll
      for (int q = 0; q < R; ++q) {
        const double s = wave_total(term[0][q] + L.term[0][q][tid + kWave]);
        if (lane == 0) L.wave[0][q][wid / 2] = s;
      }
  } else {
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int q = 0; q < R; ++q) L.term[v][q][tid] = term[v][q];
    __syncthreads();
    if (wid < W * NV * R) {
      const int v = wid / W % NV, q = wid / W / NV;
      const double* t = L.term[v][q] + tid % kBlock;
      const double s = wave_total(((t[0] + t[kBlock]) + t[2 * kBlock]) + t[3 * kBlock]);
      if (lane == 0) L.wave[v][q][wid % W] = s;
    }
  }
  __syncthreads();
  if (tid < G * NV * R) {
    const int k = tid % G, v = tid / G % NV, q = tid / G / NV;
    const int l = (blockIdx.x * R + q) * G + k;
    double s = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) s += L.wave[v][q][k * W + w];
    if (l < real) {
      const int p = slot_of(l);
      const Halves h = halves(s);
      agent_store(set + 2 * v * kResidentSlots + p, tag | h.lo);
      agent_store(set + (2 * v + 1) * kResidentSlots + p, tag | h.hi);
    }
  }
  __syncthreads();
  double acc[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] = 0;
  for (int p = tid; p < nslots; p += kResBlock) {
    if (row_order(p) >= real) continue; // a workgroup without rows: + 0
    unsigned long long w[2 * NV];
    for (long spins = 1;; ++spins) {
      bool there = true;
#pragma unroll
      for (int k = 0; k < 2 * NV; ++k) w[k] = agent_load(set + k * kResidentSlots + p);
#pragma unroll
      for (int k = 0; k < 2 * NV; ++k) there = there && (unsigned)(w[k] >> 32) == g.phase;
      if (there || give_up(g, spins, &L.failed)) break;
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] += whole((unsigned)w[2 * v], (unsigned)w[2 * v + 1]);
  }
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const double s = wave_total(acc[v]);
    if (lane == 0) L.fin[v][wid] = s;
  }
  __syncthreads();
  if (L.failed) return false;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    out[v] = 0;
#pragma unroll
    for (int w = 0; w < kResWaves; ++w) out[v] += L.fin[v][w];
  }
  // (no barrier: the next sum writes term and wave, and fin only behind a barrier of its own)
  return true;
}

// Iterations from the state of launch_cg_* (krylov.hip) between two iterations: r, p, x, rho, rho1
// and, with the Diag preconditioner, z = invD r. Leaves that state when the stop test passes (or
// p.q = 0, max_it), after `iters` iterations, or after a multiple of `check` iterations with r.r
// below `below` or not finite.
// ex: exchange vectors of n entries over the signalling-NaN sentinel of the sync-free sweeps: a
// value is there when it is not the sentinel, so nothing waits for a store to complete before the
// sum that follows it. z in turn in ex[0] and ex[1]; Chebyshev: r in ex[2], the steps' y in ex[3..].
// An entry is cleared by its owner after a sum that all its readers reached by having read it, and
// written again only after the p.q sum in between, which settles the clearing.
// ONE: a single workgroup, the exchange vectors in LDS with barriers instead of sentinels (through
// memory an exchange inside one workgroup costs as much as between two; 14 x 11 x 9: 3.9 us an iteration with the sums of
// several workgroups and z exchanged, 2.8 with block_total and p). p itself is exchanged, in ex[0]: one
// barrier more, and neither the copies' registers (two FP64 rows a lane spilled with them) nor their operations.
// PQ: the tree of q = A p's p.q on this operand (kSumRows or kSumPairs).
// Where a row has no j-th entry, ONE (bound by its instructions: 16 wavefronts on one compute unit) multiplies two zeros,
// the value and the vector's entry past the last, and adds +0 to a sum that is never -0; a wavefront without
// rows in a round does none of its work.
template <typename T, int R, bool ONE, bool CHEB, int PQ>
__global__ void __launch_bounds__(kResBlock) k_cg_resident(int n, RBMat<T> A, const T* __restrict__ invd, T* x, T* r,
                                                            T* z, T* p, T* ex, CGState* st, GridSums g,
                                                            ResidentCheb cb, int iters, int check, double below) {
  typedef typename SfBits<T>::U U;
  constexpr int K = kResidentMaxSlots;
  __shared__ SumLds lds;
  extern __shared__ char own_ex[];
  if (st->done) return;
  double rho = st->rho, rho1 = st->rho1, rr = st->rr;
  const double crit = st->crit;
  const int max_it = st->max_it;
  int it = st->it, status = st->status, done = 0, breakdown = 0;
  g.phase = (unsigned)g.head[0];
  if (threadIdx.x == 0) lds.failed = 0;

  const int stride = ONE ? n + 1 : n; // of the exchange vectors
  // whether this wavefront has rows in round q
  auto mine = [&](int q) {
    return !ONE || __builtin_amdgcn_readfirstlane((int)(q * kResBlock + (threadIdx.x & ~(kWave - 1)))) < n;
  };
  int row[R];
  unsigned on[R];    // bit j: the row has entry j; bit 31: the row exists
  unsigned at[R][K]; // byte offset of entry j's column, or of the row itself where there is none
  T a[R][K], xv[R], rv[R], dv[R], zv[R], pv[R];
  T pc[ONE ? 1 : R][ONE ? 1 : K];
  U* const exu = reinterpret_cast<U*>(ONE ? (char*)own_ex : (char*)ex);
#pragma unroll
  for (int q = 0; q < R; ++q) {
    const int i = (blockIdx.x * R + q) * kResBlock + threadIdx.x;
    const bool in = i < n;
    row[q] = in ? i : n - 1;
    const int b = __builtin_amdgcn_readfirstlane(row[q] / kWave); // (rows past n: the last row's bundle)
    const int lane = row[q] % kWave;
    const int s0 = A.bo[b], w = A.bo[b + 1] - s0;
    on[q] = in ? 1u << 31 : 0;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      const int s = s0 + min(j, max(w - 1, 0));
      a[q][j] = T(0);
      at[q][j] = (unsigned)(ONE ? n : row[q]) * (unsigned)sizeof(T);
      if (j < w) {
        a[q][j] = A.bv[(long)s * kWave + lane];
        if (in && (A.dmask[s] >> lane & 1)) {
          on[q] |= 1u << j;
          at[q][j] = (unsigned)(row[q] + A.doff[s]) * (unsigned)sizeof(T);
        }
      }
    }
    xv[q] = x[row[q]];
    rv[q] = r[row[q]];
    dv[q] = invd[row[q]];
    pv[q] = p[row[q]];
    zv[q] = CHEB ? T(0) : z[row[q]];
  }
  auto sum = [&](int q, const T (&v)[K]) {
    T acc = 0;
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (ONE || (on[q] >> j & 1)) acc = acc + a[q][j] * v[j];
    return acc;
  };
  auto publish = [&](int e, const T (&v)[R]) {
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (on[q] >> 31) {
        if constexpr (ONE) exu[e * stride + row[q]] = SfBits<T>::bits(v[q]);
        else agent_store(exu + (size_t)e * n + row[q], SfBits<T>::bits(v[q]));
      }
  };
  auto clear = [&](int e) {
    if constexpr (ONE) return;
#pragma unroll
    for (int q = 0; q < R; ++q)
      if (on[q] >> 31) agent_store(exu + (size_t)e * n + row[q], SfBits<T>::kSentinel);
  };
  // the values of exchange vector e at row q's columns
  auto gather = [&](int e, int q, T (&out)[K]) {
    const char* src = reinterpret_cast<const char*>(exu + (size_t)e * n);
    U u[K];
    if constexpr (ONE) {
#pragma unroll
      for (int j = 0; j < K; ++j) out[j] = *reinterpret_cast<const T*>(own_ex + e * stride * sizeof(T) + at[q][j]);
      return;
    }
    for (long spins = 1;; ++spins) {
      bool there = true;
#pragma unroll
      for (int j = 0; j < K; ++j) u[j] = agent_load(reinterpret_cast<const U*>(src + at[q][j]));
#pragma unroll
      for (int j = 0; j < K; ++j) there = there && u[j] != SfBits<T>::kSentinel;
      if (there || !(on[q] >> 31) || give_up(g, spins, &lds.failed)) break;
      // (reads repeated at once hold up the very stores they wait for: Chebyshev steps of 6,000 to
      // 18,000 rows took up to three times as long)
      __builtin_amdgcn_s_sleep(16);
    }
#pragma unroll
    for (int j = 0; j < K; ++j) out[j] = SfBits<T>::value(u[j]);
  };
  if constexpr (!ONE)
#pragma unroll
    for (int q = 0; q < R; ++q)
#pragma unroll
      for (int j = 0; j < K; ++j)
        pc[q][j] = *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + at[q][j]);

  if constexpr (ONE)
    if (threadIdx.x < (CHEB ? 2 + cb.order : 2)) exu[threadIdx.x * stride + n] = 0;
  __syncthreads();
  for (int e = 0; e < (CHEB ? 2 + cb.order : 2); ++e) clear(e);
  if (CHEB) publish(2, rv);
  else if (!ONE) publish(1, zv);
  double none[1][R] = {}, s1[1];
  if (!grid_sum<kSumStream, 1, ONE, R>(g, n, none, s1, lds, true)) return;
  for (int i = 0;;) {
    const int ze = CHEB ? i & 1 : (i & 1) ^ 1; // z of this iteration's direction
    if constexpr (CHEB) {
      // ChebyshevPreconditioner::_algo2 as k_cheb_step
      T y[R], cp[R];
      double xy[1][R];
      for (int m = 0; m < cb.order; ++m) {
        const T ca = (T)cb.a[m], ccb = (T)cb.b[m];
        if (ONE && m) __syncthreads();
#pragma unroll
        for (int q = 0; q < R; ++q) {
          if (m == 0) cp[q] = y[q] = T(0);
          xy[0][q] = 0.0;
          if (!mine(q)) continue;
          T v[K];
          gather(2 + m, q, v);
          const T t = sum(q, v);
          const T e = rv[q] + T(-1) * t;
          const T zz = dv[q] * e;
          if (m == 0) {
            cp[q] = zz;
            y[q] = rv[q] + ca * cp[q];
          } else {
            cp[q] = ccb * cp[q];
            cp[q] = cp[q] + T(1) * zz;
            y[q] = y[q] + ca * cp[q];
          }
          xy[0][q] = on[q] >> 31 ? 0.0 + (double)rv[q] * (double)y[q] : 0.0;
        }
        if (m < cb.order - 1 || !ONE) publish(m == cb.order - 1 ? ze : 3 + m, y);
      }
      if (!grid_sum<kSumRows, 1, ONE, R>(g, n, xy, s1, lds, false)) return;
      for (int e = 2; e < 2 + cb.order; ++e) clear(e);
#pragma unroll
      for (int q = 0; q < R; ++q) zv[q] = y[q];
      rho1 = s1[0];
    }
    const T beta = (T)(rho1 / rho);
    T qv[R];
    double pq[1][R];
    if constexpr (ONE) {
#pragma unroll
      for (int q = 0; q < R; ++q) pv[q] = zv[q] + beta * pv[q];
      publish(0, pv);
      __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < R; ++q) {
      qv[q] = T(0);
      pq[0][q] = 0.0;
      if (!mine(q)) continue;
      T v[K];
      if constexpr (ONE) {
        gather(0, q, v);
        qv[q] = sum(q, v);
      } else {
        gather(ze, q, v);
#pragma unroll
        for (int j = 0; j < K; ++j) pc[q][j] = v[j] + beta * pc[q][j];
        pv[q] = zv[q] + beta * pv[q];
        qv[q] = sum(q, pc[q]);
      }
      pq[0][q] = on[q] >> 31 ? 0.0 + (double)pv[q] * (double)qv[q] : 0.0;
    }
    if (!grid_sum<PQ, 1, ONE, R>(g, n, pq, s1, lds, true)) return;
    clear(ze);
    if (s1[0] == 0) {
      breakdown = done = 1;
      if (blockIdx.x == 0 && threadIdx.x == 0) st->pq = s1[0];
      break;
    }
    const T al = (T)(rho1 / s1[0]);
    double rs[CHEB ? 1 : 2][R], s[CHEB ? 1 : 2];
#pragma unroll
    for (int q = 0; q < R; ++q) {
      xv[q] = xv[q] + al * pv[q];
      rv[q] = rv[q] + (-al) * qv[q];
      rs[0][q] = on[q] >> 31 ? 0.0 + (double)rv[q] * (double)rv[q] : 0.0;
      if constexpr (!CHEB) {
        zv[q] = dv[q] * rv[q];
        rs[1][q] = on[q] >> 31 ? 0.0 + (double)rv[q] * (double)zv[q] : 0.0;
      }
    }
    if (CHEB) publish(2, rv);
    else if (!ONE) publish(ze ^ 1, zv);
    if (!grid_sum<kSumStream, CHEB ? 1 : 2, ONE, R>(g, n, rs, s, lds, false)) return;
    // Iteration::stop and the scalars, as k_finalize's kFinXR / kFinXRDiag
    rho = rho1;
    ++it;
    if (it >= max_it) {
      done = 1;
    } else {
      rr = s[0];
      status = rr < crit ? 1 : 0;
      done = status;
    }
    if constexpr (!CHEB) rho1 = s[1];
    ++i;
    if (done || i >= iters || (i % check == 0 && (rr < below || !isfinite(rr)))) break;
  }
#pragma unroll
  for (int q = 0; q < R; ++q)
    if (on[q] >> 31) {
      x[row[q]] = xv[q];
      r[row[q]] = rv[q];
      z[row[q]] = zv[q];
      p[row[q]] = pv[q];
    }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->rho = rho;
    st->rho1 = rho1;
    st->rr = rr;
    st->it = it;
    st->done = done;
    st->status = status;
    st->breakdown = breakdown;
    g.head[0] = (int)g.phase;
  }
}

// One row per lane as long as the compute units hold them, then two. Two rows with the Chebyshev
// preconditioner gain nothing (80^3: 67 us against 68) and are left to the launches, as is what is
// larger: four FP32 rows per lane spill (100^3: 27 us against 30).
template <typename T>
bool resident_plan(int n, const RBMat<T>& A, int cus, int cheb_order, ResidentPlan& P) {
  if (n < 1 || n > kResidentMaxRows || !A.doff || A.pair || A.ell || A.wmax > kResidentMaxSlots ||
      cheb_order > kResidentMaxOrder)
    return false;
  // the launches' grids, whose sums these are: one bundle (or pair of bundles) per wavefront
  if (rb_blocks(n, A) != bundle_blocks_max(n)) return false;
  P.pairs = A.uni > 0 && A.uni <= kUniPairMaxSlots;
  P.exchange = 2 + cheb_order;
  P.lds = P.exchange * (n + 1) * sizeof(T);
  P.one = n <= 2 * kResBlock && P.lds <= 40 * 1024;
  if (!P.one) P.lds = 0;
  const long blocks = P.one ? 1 : std::min(cus, kResidentMaxBlocks);
  P.rows = n <= blocks * kResBlock ? 1 : 2;
  P.blocks = (n + kResBlock * P.rows - 1) / (kResBlock * P.rows);
  return n <= blocks * kResBlock * P.rows && (P.rows == 1 || P.one || cheb_order == 0);
}

template <typename T, int R, bool ONE, bool CHEB>
static const void* resident_kernel(bool pairs) {
  if constexpr (sizeof(T) == 4)
    if (pairs) return (const void*)k_cg_resident<T, R, ONE, CHEB, kSumPairs>;
  return (const void*)k_cg_resident<T, R, ONE, CHEB, kSumRows>;
}

template <typename T>
bool launch_cg_resident(hipStream_t s, const ResidentPlan& P, int n, RBMat<T> A, const T* invd, T* x, T* r, T* z, T* p,
                        T* ex, CGState* st, unsigned long long* slots, int* head, const ResidentCheb& cheb, int iters,
                        int check, double below, long spins) {
  const void* f = nullptr;
  auto pick = [&](auto rows, auto one) {
    constexpr int R = decltype(rows)::value;
    constexpr bool ONE = decltype(one)::value;
    if (P.rows == R && P.one == ONE)
      f = cheb.order > 0 ? resident_kernel<T, R, ONE, true>(P.pairs) : resident_kernel<T, R, ONE, false>(P.pairs);
  };
  pick(std::integral_constant<int, 1>{}, std::false_type{});
  pick(std::integral_constant<int, 2>{}, std::false_type{});
  pick(std::integral_constant<int, 1>{}, std::true_type{});
  pick(std::integral_constant<int, 2>{}, std::true_type{});
  GridSums g{slots, head, 0, spins};
  ResidentCheb cb = cheb;
  void* args[] = {&n, &A, &invd, &x, &r, &z, &p, &ex, &st, &g, &cb, &iters, &check, &below};
  if (hipLaunchKernel(f, dim3((unsigned)P.blocks), dim3(kResBlock), args, P.lds, s) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return true;
}

#define ALIEN_HIP_INST_RESIDENT(T)                                                                              \
  template bool resident_plan<T>(int, const RBMat<T>&, int, int, ResidentPlan&);                                \
  template bool launch_cg_resident<T>(hipStream_t, const ResidentPlan&, int, RBMat<T>, const T*, T*, T*, T*, T*, \
                                      T*, CGState*, unsigned long long*, int*, const ResidentCheb&, int, int,   \
                                      double, long);
ALIEN_HIP_INST_RESIDENT(double)
ALIEN_HIP_INST_RESIDENT(float)

} // namespace alien_hip
