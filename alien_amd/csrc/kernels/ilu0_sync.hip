// ILU(0) factorisation and triangular sweeps over CSR arrays and level-set schedules, one launch
// each instead of one per level (ilu0.hip): the level order is cut into chunks of 64 rows, taken by
// waves from an atomic ticket, and each lane waits for the rows its own reads, in the order in which
// it uses them. A chunk may span levels: a lane whose rows are there goes on while others of its
// wavefront wait, so the earliest row not done yet is never held up, and every row only waits on
// earlier ones of the order. The operations of a row are those of the level kernels in their order.
// Bound by one store-to-load trip between compute units per level: 1.9 us (sweeps) and 2.4 us
// (factorisation) at 64^3, 7-point, 190 levels, where a launch per level took 4.8 and 16 us; together
// 4.69 -> 1.21 ms. Waiting for a row's entries in turn, and looking its matches up after the wait,
// took 2.9 and 19 us per level.
// Waits are bounded; one that runs out raises a flag, and a wavefront then does in order what is
// left. Matrices whose rows update more than their pivots are factorised a wavefront per row (k_sync_factor_rows).
#include "../alien_hip_internal.h"
#include "../alien/hip/HIPContext.h"
#include "device_common.h"
#include "launch.h"
#include "sync_free.h"

#include <algorithm>

namespace alien_hip {

namespace {
template <typename U>
__device__ __forceinline__ U agent_load(const U* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename U>
__device__ __forceinline__ void agent_store(U* p, U v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
typedef SfBits<double> B;
typedef B::U U;
} // namespace

// out = sentinel; work: ticket and flag, cleared
__global__ void __launch_bounds__(kBlock) k_sync_fill(int n, double* out, int* work) {
  for (long i = (long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock)
    reinterpret_cast<U*>(out)[i] = B::kSentinel;
  if (blockIdx.x == 0 && threadIdx.x < 2) work[threadIdx.x] = 0;
}

__device__ __forceinline__ int next_chunk(int* ticket) {
  int c = 0;
  if ((threadIdx.x & (kWave - 1)) == 0) c = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __builtin_amdgcn_readfirstlane(c);
}
// one more poll without result: true when the wait is over
__device__ __forceinline__ bool wait_over(long& spins, long limit, int* flag) {
  if (++spins <= limit && ((spins & 255) != 0 || agent_load(flag) == 0)) {
    __builtin_amdgcn_s_sleep(2);
    return false;
  }
  agent_store(flag, 1);
  return true;
}

// Row i of the factorisation (k_ilu0_factor_level), all rows it reads being done: their pivots in
// piv, their entries read past the caches. Its own strictly-upper entries change only where a column
// of a lower row is its own too; piv is then published after those have landed.
__device__ __forceinline__ void factor_row(int i, const int* __restrict__ ro, const int* __restrict__ cols,
                                           const int* __restrict__ dcol, double* lu, double* piv) {
  const int rb = ro[i], re = ro[i + 1], di = dcol[i];
  bool upper = false;
  double d = lu[di];
  for (int k = rb; k < di; ++k) {
    const int kr = cols[k];
    const double aik = lu[k] / B::value(agent_load(reinterpret_cast<const U*>(piv) + kr));
    lu[k] = aik;
    int p = ro[kr];
    const int pe = ro[kr + 1];
    for (int j = k + 1; j < re; ++j) {
      const int cj = cols[j];
      while (p < pe && cols[p] < cj) ++p;
      if (p == pe) break;
      if (cols[p] == cj) {
        const double akj = B::value(agent_load(reinterpret_cast<const U*>(lu) + p));
        if (j == di) {
          d = d - aik * akj;
        } else if (j < di) {
          lu[j] = lu[j] - aik * akj;
        } else {
          upper = true;
          U* e = reinterpret_cast<U*>(lu) + j;
          agent_store(e, B::bits(B::value(agent_load(e)) - aik * akj));
        }
      }
    }
  }
  lu[di] = d;
  if (upper) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  agent_store(reinterpret_cast<U*>(piv) + i, B::bits(d));
}

// Rows of at most kSyncSlots entries to wait for read them all in each poll (one trip when the last
// is there, where waiting for one after the other takes a trip each); longer rows wait in turn.
constexpr int kSyncSlots = 8;

// A short row whose only entry that its lower rows' entries touch is its diagonal (every 7-point
// row): the entries' positions are looked up before the wait, and after it all rows' values are read
// at once: pivot d - sum (a_ik / u_kk) a_ki. Other rows run factor_row.
struct ShortFactor {
  int at[kSyncSlots];  // a_ki in row k, -1: none
  double l[kSyncSlots];
  bool plain;
};
__device__ __forceinline__ void look_up(ShortFactor& f, int i, int rb, int di, int re, const int* __restrict__ ro,
                                        const int* __restrict__ cols, const int* __restrict__ dcol,
                                        const double* __restrict__ lu, const int (&col)[kSyncSlots]) {
  f.plain = di - rb <= kSyncSlots;
#pragma unroll
  for (int s = 0; s < kSyncSlots; ++s) {
    f.at[s] = -1;
    f.l[s] = 0;
    if (!f.plain || rb + s >= di) continue;
    f.l[s] = lu[rb + s];
    const int pe = ro[col[s] + 1];
    for (int p = dcol[col[s]] + 1; p < pe; ++p) {
      const int c = cols[p];
      if (c == i) f.at[s] = p;
      else
        for (int j = rb + s + 1; j < re; ++j) f.plain = f.plain && cols[j] != c;
    }
  }
}

// As k_sync_fill before a factorisation; work[2]: whether more than an eighth of 256 rows spread over the matrix are not
// plain ones, by the nearest row that each reads. It chooses between two kernels that take any row (a host that chose
// would have to read the matrix back).
constexpr int kSyncSample = kBlock;
__global__ void __launch_bounds__(kBlock) k_sync_factor_start(int n, const int* __restrict__ ro,
                                                               const int* __restrict__ cols, const int* __restrict__ dcol,
                                                               double* piv, int* work) {
  for (long i = (long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock)
    reinterpret_cast<U*>(piv)[i] = B::kSentinel;
  if (blockIdx.x != 0) return;
  const int sample = min(n, kSyncSample);
  bool other = false;
  if ((int)threadIdx.x < sample) {
    const int i = (int)((long)threadIdx.x * n / sample), rb = ro[i], di = dcol[i], re = ro[i + 1];
    const int near = di > rb ? cols[di - 1] : -1;
    other = di - rb > kSyncSlots;
    if (near >= 0)
      for (int p = dcol[near] + 1, pe = ro[near + 1]; p < pe; ++p)
        for (int j = di + 1, c = cols[p]; j < re; ++j) other = other || cols[j] == c;
  }
  const int others = __syncthreads_count(other);
  if (threadIdx.x < 2) work[threadIdx.x] = 0;
  if (threadIdx.x == 2) work[2] = 8 * others > sample;
}

__global__ void __launch_bounds__(kBlock) k_sync_factor(int n, const int* __restrict__ rows,
                                                         const int* __restrict__ ro, const int* __restrict__ cols,
                                                         const int* __restrict__ dcol, double* lu, double* piv,
                                                         int* work, long limit) {
  if (work[2]) return;
  const int lane = threadIdx.x & (kWave - 1);
  const U* pv = reinterpret_cast<const U*>(piv);
  for (int c; (long)(c = next_chunk(work)) * kWave < n;) {
    const long q = (long)c * kWave + lane;
    bool open = q < n;
    const int i = open ? rows[q] : 0;
    const int rb = open ? ro[i] : 0, di = open ? dcol[i] : 0, re = open ? ro[i + 1] : 0;
    int k = rb;
    int col[kSyncSlots];
#pragma unroll
    for (int s = 0; s < kSyncSlots; ++s) col[s] = rb + s < di ? cols[rb + s] : -1;
    ShortFactor f;
    look_up(f, i, rb, di, re, ro, cols, dcol, lu, col);
    double d = open ? lu[di] : 0;
    long spins = 0;
    while (__any(open)) {
      if (!open) continue;
      if (f.plain) {
        U b[kSyncSlots];
        bool there = true;
#pragma unroll
        for (int s = 0; s < kSyncSlots; ++s)
          if (col[s] >= 0) b[s] = agent_load(pv + col[s]);
#pragma unroll
        for (int s = 0; s < kSyncSlots; ++s) there = there && (col[s] < 0 || b[s] != B::kSentinel);
        if (there) {
          double t[kSyncSlots];
#pragma unroll
          for (int s = 0; s < kSyncSlots; ++s)
            if (f.at[s] >= 0) t[s] = B::value(agent_load(reinterpret_cast<const U*>(lu) + f.at[s]));
#pragma unroll
          for (int s = 0; s < kSyncSlots; ++s)
            if (col[s] >= 0) f.l[s] = f.l[s] / B::value(b[s]);
#pragma unroll
          for (int s = 0; s < kSyncSlots; ++s)
            if (f.at[s] >= 0) d = d - f.l[s] * t[s];
          agent_store(reinterpret_cast<U*>(piv) + i, B::bits(d));
#pragma unroll
          for (int s = 0; s < kSyncSlots; ++s)
            if (col[s] >= 0) lu[rb + s] = f.l[s];
          lu[di] = d;
          open = false;
          continue;
        }
      } else {
        while (k < di && agent_load(pv + cols[k]) != B::kSentinel) ++k;
        if (k >= di) {
          factor_row(i, ro, cols, dcol, lu, piv);
          open = false;
          continue;
        }
      }
      if (wait_over(spins, limit, work + 1)) open = false;
    }
  }
}

// A row by a wavefront, an entry per lane, for matrices whose rows are mostly not plain: a lane that merges the rows of one
// of its own alone takes 150 us a row of 27 entries, as in the level kernels, and the lanes of a wavefront whose rows
// become ready at different times take turns at that. Per lower entry, in order: the entries to its right of
// that column's row, found by comparing columns across the lanes (the next such row's are asked for meanwhile), and
// one trip for their values. `per` rows a ticket. Rows of more entries than lanes are left to one lane (factor_row).
// Bound by that chain, about 1 us a lower entry. Launches per level, lanes as in k_sync_factor, this: 27-point 40^3 45.6,
// 63.5, 4.8 ms; 9-point 400 x 400 22.6, 26.9, 5.4; 20,000 rows of 41 entries, 1000 levels, 267, 4760 (waits given up), 29.
__device__ __forceinline__ double of_lane(double v, int lane) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)b, lane), hi = __builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
  return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}
__global__ void __launch_bounds__(kBlock) k_sync_factor_rows(int n, int per, const int* __restrict__ rows,
                                                              const int* __restrict__ ro, const int* __restrict__ cols,
                                                              const int* __restrict__ dcol, double* lu, double* piv,
                                                              int* work, long limit) {
  if (!work[2]) return;
  const int lane = threadIdx.x & (kWave - 1);
  const U* pv = reinterpret_cast<const U*>(piv);
  U* lv = reinterpret_cast<U*>(lu);
  for (int c; (long)(c = next_chunk(work)) * per < n;) {
    const long end = min((long)n, ((long)c + 1) * per);
    for (long q = (long)c * per; q < end; ++q) {
      const int i = rows[q], rb = ro[i], di = dcol[i], re = ro[i + 1];
      bool there = true;
      for (int k0 = rb; k0 < di && there; k0 += kWave) {
        const bool on = k0 + lane < di;
        const int col = on ? cols[k0 + lane] : 0;
        long spins = 0;
        while (there && __any(on && agent_load(pv + col) == B::kSentinel)) there = !wait_over(spins, limit, work + 1);
      }
      if (!there) continue; // given up, not touched
      if (re - rb > kWave) {
        if (lane == 0) factor_row(i, ro, cols, dcol, lu, piv);
        continue;
      }
      const int low = di - rb, j = rb + lane;
      const bool has = j < re;
      const int cj = has ? cols[j] : -1;
      double v = has ? lu[j] : 0.0;
      int ub = 0, ue = 0; // of a lower entry's lane: the entries of its column's row beyond the diagonal
      double pk = 1.0;    // and that row's pivot
      if (lane < low) {
        ub = dcol[cj] + 1;
        ue = ro[cj + 1];
        pk = B::value(agent_load(pv + cj));
      }
      auto column = [&](int t, int p0) { // this lane's of those entries, from p0 on
        const int p = p0 + lane;
        return p < __builtin_amdgcn_readlane(ue, t) ? cols[p] : -2;
      };
      bool touched = false;
      int cp = low > 0 ? column(0, __builtin_amdgcn_readlane(ub, 0)) : -2;
      for (int t = 0; t < low; ++t) {
        const int b = __builtin_amdgcn_readlane(ub, t), e = __builtin_amdgcn_readlane(ue, t);
        const double a = of_lane(v, t) / of_lane(pk, t);
        if (lane == t) v = a;
        int at = -1;
        for (int p0 = b; p0 < e; p0 += kWave) {
          if (p0 > b) cp = column(t, p0);
          const int m = min(e - p0, kWave);
          for (int u = 0; u < m; ++u)
            if (lane > t && cj == __builtin_amdgcn_readlane(cp, u)) at = p0 + u;
        }
        if (t + 1 < low) cp = column(t + 1, __builtin_amdgcn_readlane(ub, t + 1));
        if (at >= 0) {
          v = v - a * B::value(agent_load(lv + at));
          touched = true;
        }
      }
      if (has && lane <= low) lu[j] = v;
      const bool out = has && lane > low && touched;
      if (out) agent_store(lv + j, B::bits(v));
      if (__any(out)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == low) agent_store(reinterpret_cast<U*>(piv) + i, B::bits(v));
    }
  }
}

template <bool UPPER>
__global__ void __launch_bounds__(kBlock) k_sync_sweep(int n, const int* __restrict__ rows,
                                                        const int* __restrict__ ro, const int* __restrict__ cols,
                                                        const int* __restrict__ dcol, const double* __restrict__ lu,
                                                        const double* in, double* out, int* work, long limit) {
  const int lane = threadIdx.x & (kWave - 1);
  U* o = reinterpret_cast<U*>(out);
  for (int c; (long)(c = next_chunk(work)) * kWave < n;) {
    const long q = (long)c * kWave + lane;
    bool open = q < n;
    const int i = open ? rows[q] : 0;
    const int d = open ? dcol[i] : 0;
    int k = open ? (UPPER ? d + 1 : ro[i]) : 0;
    const int e = open ? (UPPER ? ro[i + 1] : d) : 0;
    double v = open ? in[i] : 0;
    const double diag = open && UPPER ? lu[d] : 1.0;
    const bool few = e - k <= kSyncSlots;
    int col[kSyncSlots];
    double a[kSyncSlots];
#pragma unroll
    for (int s = 0; s < kSyncSlots; ++s) {
      const bool on = few && k + s < e;
      col[s] = on ? cols[k + s] : -1;
      a[s] = on ? lu[k + s] : 0;
    }
    long spins = 0;
    while (__any(open)) {
      if (!open) continue;
      bool there = true;
      if (few) {
        U b[kSyncSlots];
#pragma unroll
        for (int s = 0; s < kSyncSlots; ++s)
          if (col[s] >= 0) b[s] = agent_load(o + col[s]);
#pragma unroll
        for (int s = 0; s < kSyncSlots; ++s) there = there && (col[s] < 0 || b[s] != B::kSentinel);
        if (there)
#pragma unroll
          for (int s = 0; s < kSyncSlots; ++s)
            if (col[s] >= 0) v = v - a[s] * B::value(b[s]);
      } else {
        while (k < e) {
          const U b = agent_load(o + cols[k]);
          if (b == B::kSentinel) break;
          v = v - lu[k] * B::value(b);
          ++k;
        }
        there = k >= e;
      }
      if (there) {
        if (UPPER) v = v / diag;
        agent_store(o + i, B::bits(v));
        open = false;
      } else if (wait_over(spins, limit, work + 1)) {
        open = false;
      }
    }
  }
}

// After a wait that ran out of polls: the rows left, in order (one lane; without the flag it returns
// at once). A row given up has not been touched.
__global__ void __launch_bounds__(kWave) k_sync_factor_rest(int n, const int* rows, const int* ro, const int* cols,
                                                             const int* dcol, double* lu, double* piv, int* work) {
  if (agent_load(work + 1) == 0) return;
  if (threadIdx.x == 0)
    for (int q = 0; q < n; ++q)
      if (agent_load(reinterpret_cast<const U*>(piv) + rows[q]) == B::kSentinel)
        factor_row(rows[q], ro, cols, dcol, lu, piv);
}
template <bool UPPER>
__global__ void __launch_bounds__(kWave) k_sync_sweep_rest(int n, const int* rows, const int* ro, const int* cols,
                                                            const int* dcol, const double* lu, const double* in,
                                                            double* out, int* work) {
  if (agent_load(work + 1) == 0) return;
  U* o = reinterpret_cast<U*>(out);
  if (threadIdx.x == 0)
    for (int q = 0; q < n; ++q) {
      const int i = rows[q], d = dcol[i];
      if (agent_load(o + i) != B::kSentinel) continue;
      double v = in[i];
      const int e = UPPER ? ro[i + 1] : d;
      for (int k = UPPER ? d + 1 : ro[i]; k < e; ++k) v = v - lu[k] * B::value(agent_load(o + cols[k]));
      agent_store(o + i, B::bits(UPPER ? v / lu[d] : v));
    }
}

// Polls of a wait here: a row may wait for all of the thousands taken before it, each taking as long as its
// entries make it (with the level-ordered sweeps' number of polls 20,000 rows of 41 entries gave up and took 4.8 s).
static long sync_spins() { return 64 * g_ilu_sf_spins; }

// Lanes for about ten levels' rows (a row's entries are looked up ahead of its turn), 64 to 256
// workgroups, never more waves than chunks; ALIEN_HIP_ILU_SF_BLOCKS overrides. Factorisation and solve
// of the 7-point 96^3 matrix: 2.58 ms with 48 workgroups, 2.31 with 64, 2.12 with 128, 2.22 with 192;
// 64^3: 1.37 with 32, 1.21 with 64 or 96, 1.34 with 192.
static dim3 sync_grid(int n, int nlevels) {
  const long avg = n / std::max(1, nlevels);
  long blocks = std::min(256L, std::max(64L, (10 * avg + kBlock - 1) / kBlock));
  if (g_ilu_sf_blocks > 0) blocks = g_ilu_sf_blocks;
  const long chunks = ((long)n + kWave - 1) / kWave, waves = kBlock / kWave;
  return dim3((unsigned)std::max(1L, std::min(blocks, (chunks + waves - 1) / waves)));
}

// Levels of more rows than this on average are launched one by one (few, and each fills the device). 2,000,000 rows of
// three entries, a launch each and one launch, us, by rows a level: 12,000 factorisation 621 and 410, solve 1007 and 770;
// 16,000 470 and 409, 752 and 771; 20,000 386 and 407, 611 and 767; 32,000 254 and 406, 398 and 764.
constexpr long kSyncAvgRows = 16384;
bool sync_levels(int n, int nlevels) {
  return g_ilu_sync_free && nlevels > 2 && n > 0 && n <= std::min(g_ilu_sf_avg_rows, kSyncAvgRows) * nlevels;
}

void launch_sync_factor(hipStream_t st, int n, int nlevels, const int* rows, const int* ro, const int* cols,
                        const int* dcol, double* lu, double* piv, int* work) {
  hipLaunchKernelGGL(k_sync_factor_start, dim3(grid_for(n, 4)), dim3(kBlock), 0, st, n, ro, cols, dcol, piv,
                     work);
  hipLaunchKernelGGL(k_sync_factor, sync_grid(n, nlevels), dim3(kBlock), 0, st, n, rows, ro, cols, dcol, lu, piv, work,
                     sync_spins());
  // a wavefront per row of about ten levels, 256 to 2048 of them
  const long avg = n / std::max(1, nlevels), waves = kBlock / kWave;
  const int per = (int)std::min(16L, std::max(1L, avg / 2048));
  const long blocks = std::min((10 * avg / per + waves - 1) / waves, 512L), most = ((long)n / per + waves) / waves;
  hipLaunchKernelGGL(k_sync_factor_rows, dim3((unsigned)std::max(1L, std::min(std::max(blocks, 64L), most))), dim3(kBlock), 0,
                     st, n, per, rows, ro, cols, dcol, lu, piv, work, sync_spins());
  hipLaunchKernelGGL(k_sync_factor_rest, dim3(1), dim3(kWave), 0, st, n, rows, ro, cols, dcol, lu, piv, work);
}

template <bool UPPER>
static void sync_sweep(hipStream_t st, int n, int nlevels, const int* rows, const int* ro, const int* cols,
                       const int* dcol, const double* lu, const double* in, double* out, int* work) {
  hipLaunchKernelGGL(k_sync_fill, dim3(grid_for(n, 4)), dim3(kBlock), 0, st, n, out, work);
  hipLaunchKernelGGL(k_sync_sweep<UPPER>, sync_grid(n, nlevels), dim3(kBlock), 0, st, n, rows, ro, cols, dcol, lu, in,
                     out, work, sync_spins());
  hipLaunchKernelGGL(k_sync_sweep_rest<UPPER>, dim3(1), dim3(kWave), 0, st, n, rows, ro, cols, dcol, lu, in, out, work);
}

void launch_sync_solve(hipStream_t st, int n, int nl, const int* lrows, int nu, const int* urows, const int* ro,
                       const int* cols, const int* dcol, const double* lu, const double* y, double* t, double* x,
                       int* work) {
  sync_sweep<false>(st, n, nl, lrows, ro, cols, dcol, lu, y, t, work);
  sync_sweep<true>(st, n, nu, urows, ro, cols, dcol, lu, t, x, work);
}

} // namespace alien_hip
