// ILU(0) of full 7-point matrices on lexicographic grids, in pencils of 8 x 8 grid lines.
//
// The level-set sweeps (ilu0.hip) pay one trip between compute units per level: i + j + k levels,
// 382 at 128^3, about 1.8 us each. Here a wavefront owns the 64 grid lines of an 8 x 8 pencil,
// lane (yl, zl) marches along x with a skew of yl + zl steps, and so meets each neighbour inside
// the pencil one step behind it: the own line's in a register, the others' by lane exchange. Only
// the values on two faces travel to the next pencils, ny / 8 + nz / 8 - 2 trips in a row (30 at
// 128^3). Measured there in FP64, against the sync-free level sweeps: lower sweep 115 us (653),
// upper 133 us (667), factorisation 204 us (382 launches, 7.5 ms), and no level sets to build on
// the host (21 ms); BiCGStab to 1e-8, 8 iterations, set-up included: 53.1 -> 9.3 ms.
//
// Storage ("skewed"): step s of pencil p holds the 64 values of its lanes contiguously at
// (p * steps + s) * 64 + lane, x = s - yl - zl; a step's operands are coalesced loads, and the
// lower sweep's result is left in the order in which the upper sweep (the same steps backwards)
// reads it. Steps outside a line are padding, (nx + 14) / nx and the last pencils' missing lines.
//
// Which rows exist is geometry: the plan is taken only where every row holds exactly its in-grid
// neighbours (launch_pencil_check), so rows couple only cells of opposite parity, the one update
// of the IKJ factorisation (ILU0Preconditioner.h:157-177) that finds a match is the pivot's own,
// u_ii -= (a_ik / u_kk) a_ki, and the strictly-upper entries stay A's. Each row does the
// operations of the sequential code in its order (ascending columns: z-, y-, x-, then x+, y+, z+;
// an absent neighbour does none), so factor and sweeps are its results bit for bit.
#include "../alien_hip_internal.h"
#include "../alien/hip/HIPContext.h"
#include "device_common.h"
#include "launch.h"
#include "sync_free.h"

namespace alien_hip {

constexpr int kPen = 8;         // lines of a pencil per direction
constexpr int kPenChunk = 8;    // steps whose operands are loaded together
constexpr int kPenSkew = 2 * (kPen - 1);
static_assert(kPen * kPen == kWave && kPen * kPenChunk == kWave, "a face's chunk is one load of the wavefront");

bool pencil_grid(int n, const int* ro, const int* cols, PencilGrid& g) {
  if (n < 8 || ro[1] - ro[0] != 4 || cols[0] != 0 || cols[1] != 1) return false;
  const int s2 = cols[2], s3 = cols[3];
  if (s2 < 2 || s3 % s2 != 0 || n % s3 != 0) return false;
  g.nx = s2;
  g.ny = s3 / s2;
  g.nz = n / s3;
  if (g.ny < 2 || g.nz < 2) return false;
  const long nx = g.nx, ny = g.ny, nz = g.nz;
  if ((long)ro[n] != 7L * n - 2 * (nx * ny + ny * nz + nz * nx)) return false;
  g.py = (g.ny + kPen - 1) / kPen;
  g.pz = (g.nz + kPen - 1) / kPen;
  g.steps = (g.nx + kPenSkew + kPenChunk - 1) / kPenChunk * kPenChunk;
  // thin grids are left to the level sets: at 8 positions a row the arrays take 0.5 KB a row, theirs 0.16
  return g.positions() <= 8L * n && g.positions() <= 0x7fffffffL;
}

std::vector<int> pencil_order(const PencilGrid& g) {
  std::vector<int> o;
  o.reserve(g.pencils());
  for (int d = 0; d <= g.py + g.pz - 2; ++d)
    for (int c = std::max(0, d - g.py + 1); c <= std::min(d, g.pz - 1); ++c) o.push_back(c * g.py + d - c);
  return o;
}

// *bad = 1 unless row i holds exactly the cells next to cell i in the grid
__global__ void __launch_bounds__(kBlock) k_pencil_check(int n, PencilGrid g, const int* __restrict__ ro,
                                                          const int* __restrict__ cols, int* bad) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int s3 = g.nx * g.ny, x = i % g.nx, y = i / g.nx % g.ny, z = i / s3;
  const int at[7] = {i - s3, i - g.nx, i - 1, i, i + 1, i + g.nx, i + s3};
  const bool on[7] = {z > 0, y > 0, x > 0, true, x < g.nx - 1, y < g.ny - 1, z < g.nz - 1};
  int k = ro[i];
  const int e = ro[i + 1];
  bool ok = true;
#pragma unroll
  for (int q = 0; q < 7; ++q)
    if (on[q]) {
      ok = ok && k < e && cols[k] == at[q];
      ++k;
    }
  if (!ok || k != e) *bad = 1;
}

// The seven diagonals of A in skewed order (base + q * positions, q = z-, y-, x-, diagonal, x+, y+,
// z+; 0 where a cell has no such neighbour), and per lower neighbour k of row i the entry a_ki
// (trans + q * positions).
__global__ void __launch_bounds__(kBlock) k_pencil_fill(PencilGrid g, const int* __restrict__ ro,
                                                         const double* __restrict__ vals, double* __restrict__ base,
                                                         double* __restrict__ trans) {
  const long pos = (long)blockIdx.x * kBlock + threadIdx.x, np = g.positions();
  if (pos >= np) return;
  const int lane = (int)(pos % kWave), p = (int)(pos / kWave / g.steps), s = (int)(pos / kWave % g.steps);
  const int yl = lane % kPen, zl = lane / kPen;
  const int x = s - yl - zl, y = p % g.py * kPen + yl, z = p / g.py * kPen + zl;
  double v[7] = {0, 0, 0, 0, 0, 0, 0}, t[3] = {0, 0, 0};
  if (x >= 0 && x < g.nx && y < g.ny && z < g.nz) {
    const int s3 = g.nx * g.ny, i = z * s3 + y * g.nx + x;
    const bool xu = x < g.nx - 1, yu = y < g.ny - 1, zu = z < g.nz - 1;
    int k = ro[i];
    if (x > 0) t[2] = vals[k - 1 - (yu ? 1 : 0) - (zu ? 1 : 0)]; // row i - 1 ends with x+, y+, z+
    if (z > 0) v[0] = vals[k++], t[0] = vals[ro[i - s3 + 1] - 1];
    if (y > 0) v[1] = vals[k++], t[1] = vals[ro[i - g.nx + 1] - 1 - (zu ? 1 : 0)];
    if (x > 0) v[2] = vals[k++];
    v[3] = vals[k++];
    if (xu) v[4] = vals[k++];
    if (yu) v[5] = vals[k++];
    if (zu) v[6] = vals[k++];
  }
#pragma unroll
  for (int q = 0; q < 7; ++q) base[q * np + pos] = v[q];
#pragma unroll
  for (int q = 0; q < 3; ++q) trans[q * np + pos] = t[q];
}

// The factor in CSR order, from its skewed storage (lu: A's values on entry)
__global__ void __launch_bounds__(kBlock) k_pencil_to_csr(int n, PencilGrid g, const int* __restrict__ ro,
                                                           const double* __restrict__ base, double* __restrict__ lu) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int x = i % g.nx, y = i / g.nx % g.ny, z = i / (g.nx * g.ny);
  const long np = g.positions(), pos = g.position(x, y, z);
  int k = ro[i];
  if (z > 0) lu[k++] = base[pos];
  if (y > 0) lu[k++] = base[np + pos];
  if (x > 0) lu[k++] = base[2 * np + pos];
  lu[k] = base[3 * np + pos];
}

__global__ void __launch_bounds__(kBlock) k_pencil_demote(long n, const double* __restrict__ a, float* __restrict__ b) {
  for (long i = (long)blockIdx.x * kBlock + threadIdx.x; i < n; i += (long)gridDim.x * kBlock) b[i] = (float)a[i];
}
template <typename T>
__global__ void __launch_bounds__(kBlock) k_pencil_init(long nhalo, T* halo, int* work) {
  typedef typename SfBits<T>::U U;
  for (long i = (long)blockIdx.x * kBlock + threadIdx.x; i < nhalo; i += (long)gridDim.x * kBlock)
    reinterpret_cast<U*>(halo)[i] = SfBits<T>::kSentinel;
  if (blockIdx.x == 0 && threadIdx.x < kPencilWork) work[threadIdx.x] = 0;
}

// The value of the lane one line back in y (lower; one ahead: upper), within rows of 16 lanes
template <bool UPPER>
__device__ __forceinline__ unsigned dpp_y(unsigned v) {
  return (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, UPPER ? 0x101 : 0x111, 0xf, 0xf, true);
}
template <bool UPPER>
__device__ __forceinline__ float lane_y(float v) {
  return __uint_as_float(dpp_y<UPPER>(__float_as_uint(v)));
}
template <bool UPPER>
__device__ __forceinline__ double lane_y(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned long long lo = dpp_y<UPPER>((unsigned)b), hi = dpp_y<UPPER>((unsigned)(b >> 32));
  return __longlong_as_double((long long)(hi << 32 | lo));
}

// One sweep: kPenLower t = L^-1 in, kPenUpper out = U^-1 t, kPenFactor the factorisation (lower and
// diagonal arrays of F updated in place). A wavefront per pencil, taken from a ticket in an order
// in which every pencil comes after those it reads, so a wavefront waits only on wavefronts that
// are running. Face values go out as agent-scope relaxed stores over a signalling-NaN sentinel (as
// in the sync-free level sweeps: no flag, a value is there when it is not the sentinel) and come in
// one load per face and chunk, issued a chunk ahead and polled again only if it came too early.
// Two sets of faces and tickets: the lower sweep uses set 0 and clears set 1, the upper sweep and
// the factorisation the other way round, so neither needs a clearing launch before it. Waits are
// bounded (limit polls); one that runs out raises work[2], in the upper sweep work[3], and the redo kernel
// follows. The upper sweep stores nothing after a lower one that gave up: `out` may be `in`, which the redo then reads.
// Bound by the instructions and waits of a lone wavefront, 0.12 us a lower step and 0.17 an upper one (a lane
// exchange, three dependent subtractions, the upper's division), and per trip between pencils by 15 steps of skew
// and chunk and 1.6 us from store to load. Operands of a step of the next chunk are loaded during each lane exchange, at
// a scalar address + lane + constant, into the other of two register sets: nothing waits for a load before its
// step (copying or polling beside them waited for all: 156 and 171 us). The upper sweep's results go out 8 x of 8 lines
// a store from LDS (64 lines a store, 8 bytes each: 165 us). Tried: the exchange in the vector unit (row rotation,
// permlane swaps) in place of ds_bpermute, 142 against 117 us.
enum PencilSweep { kPenLower = 0, kPenUpper = 1, kPenFactor = 2 };
template <typename T, int KIND>
__global__ void __launch_bounds__(kWave) k_pencil_sweep(PencilFactor<T> F, const double* __restrict__ trans,
                                                         const T* __restrict__ in, T* __restrict__ out, long limit,
                                                         const int* __restrict__ done) {
  if (done && *done) return;
  typedef typename SfBits<T>::U U;
  constexpr bool UP = KIND == kPenUpper, FAC = KIND == kPenFactor;
  constexpr int set = KIND == kPenLower ? 0 : 1;
  constexpr int C = kPenChunk;
  const PencilGrid& g = F.g;
  const int np = g.pencils(), S = g.steps;
  const int lane = threadIdx.x, yl = lane % kPen, zl = lane / kPen;
  __shared__ T face[3][kWave], val[C][kWave]; // face[2]: zeros
  int* err = F.work + (UP ? 3 : 2);

  int tk = 0;
  if (lane == 0) tk = __hip_atomic_fetch_add(F.work + set, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  tk = __builtin_amdgcn_readfirstlane(tk);
  if (tk >= np) return;
  const int p = __builtin_amdgcn_readfirstlane(F.order[UP ? np - 1 - tk : tk]);
  const int b = p % g.py, c = p / g.py;
  const int y = b * kPen + yl, z = c * kPen + zl;
  const bool rowok = y < g.ny && z < g.nz;
  const long npos = g.positions();
  const long base = (long)p * S * kWave; // uniform: a step's operand is at a scalar address + the lane + a constant
  const long line = rowok ? ((long)z * g.ny + y) * g.nx : 0;
  const bool hasy = UP ? y < g.ny - 1 : y > 0, hasz = UP ? z < g.nz - 1 : z > 0;
  // z, y, x neighbour's coefficient (the sweep's own triangle)
  T* az = F.base + (UP ? 6 : 0) * npos + base;
  T* ay = F.base + (UP ? 5 : 1) * npos + base;
  T* ax = F.base + (UP ? 4 : 2) * npos + base;
  T* dd = F.base + 3 * npos + base;
  T* tt = F.t + base;
  constexpr int dir = UP ? -kWave : kWave; // from step to step

  U* halo = reinterpret_cast<U*>(F.halo) + set * g.halo();
  U* hy = halo;                         // y faces
  U* hz = halo + g.halo() / 2;          // z faces
  {
    U* other = reinterpret_cast<U*>(F.halo) + (1 - set) * g.halo();
    for (int k = lane; k < S * kPen; k += kWave) {
      other[(long)p * S * kPen + k] = SfBits<T>::kSentinel;
      other[g.halo() / 2 + (long)p * S * kPen + k] = SfBits<T>::kSentinel;
    }
    if (tk == 0 && lane == 0) F.work[1 - set] = 0;
  }
  if (UP && __hip_atomic_load(F.work + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) return;
  const bool fromy = UP ? b < g.py - 1 : b > 0, fromz = UP ? c < g.pz - 1 : c > 0; // a pencil feeds this one
  const bool toy = UP ? b > 0 : b < g.py - 1, toz = UP ? c > 0 : c < g.pz - 1;     // this one feeds a pencil
  constexpr int edge = UP ? kPen - 1 : 0, far = kPen - 1 - edge; // lines fed by, and feeding, another pencil
  // this lane's part in a face's chunk: step fj of it, line fk
  const int fj = lane / kPen, fk = lane % kPen;
  const U* yfrom = hy + (long)(fromy ? (UP ? p + 1 : p - 1) : p) * S * kPen; // (a pencil's own where none feeds it: not used)
  const U* zfrom = hz + (long)(fromz ? (UP ? p + g.py : p - g.py) : p) * S * kPen;
  U* yto = hy + (long)p * S * kPen;
  U* zto = hz + (long)p * S * kPen;
  const bool line_y = fromy && c * kPen + fk < g.nz, line_z = fromz && b * kPen + fk < g.ny; // the fed line exists
  auto step = [&](int s) { return UP ? S - 1 - s : s; };
  // Loads and stores of the march are unconditional (lanes without one use a place of their own):
  // memory operations complete in order, and behind a branch the compiler would wait for all of them.
  struct Face {
    U y, z;
    bool ny, nz; // needed
  };
  auto face_load = [&](int s0, Face& f) {
    const int s = step(s0 + fj);
    const bool in_x = (unsigned)(s - edge - fk) < (unsigned)g.nx;
    f.ny = line_y && in_x;
    f.nz = line_z && in_x;
    const unsigned o = (unsigned)min(max(s + far - edge, 0), S - 1) * kPen + fk;
    f.y = __hip_atomic_load(yfrom + o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    f.z = __hip_atomic_load(zfrom + o, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  struct Ops {
    T z[C], y[C], x[C], r[C], d[C];
    T tz[FAC ? C : 1], ty[FAC ? C : 1], tx[FAC ? C : 1];
  };
  // step s0 + j's operands; u: step(s0) * kWave, xc: the lane's x at s0
  auto fetch = [&](long u, int xc, int j, Ops& o) {
    const int q = j * dir;
    o.z[j] = (az + u + lane)[q];
    o.y[j] = (ay + u + lane)[q];
    o.x[j] = (ax + u + lane)[q];
    if constexpr (KIND == kPenLower) o.r[j] = in[line + min(max(xc + j, 0), g.nx - 1)];
    if constexpr (UP) o.r[j] = (tt + u + lane)[q];
    if constexpr (UP || FAC) o.d[j] = (dd + u + lane)[q];
    if constexpr (FAC) {
      o.tz[j] = (trans + base + u + lane)[q];
      o.ty[j] = (trans + npos + base + u + lane)[q];
      o.tx[j] = (trans + 2 * npos + base + u + lane)[q];
    }
  };

  T own = T(0);
  Face fc;
  // a lane takes the face's value, or 0 for want of a neighbour, in place of another lane's
  const bool face_lane_y = yl == edge || !hasy, face_lane_z = zl == edge || !hasz;
  const T* face_y = &face[yl == edge && hasy ? 0 : 2][zl];
  const T* face_z = &face[zl == edge && hasz ? 1 : 2][yl];
  face[2][lane] = T(0);
  // the steps s0 .. s0 + C - 1 on their operands o; o_next: those of the chunk at `ahead`
  auto march = [&](int s0, const Ops& o, int ahead, Ops& o_next) {
    // A first look that waits for the faces alone, then the polls: one loop for both would wait, each time, for
    // every load issued since (the next chunk's operands).
    auto missing = [&] {
      return __any(((int)fc.ny & (int)(fc.y == SfBits<T>::kSentinel)) | ((int)fc.nz & (int)(fc.z == SfBits<T>::kSentinel)));
    };
    if (missing()) {
      long spins = 0;
      do {
        if (++spins > limit) {
          if (lane == 0) __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        if ((spins & 255) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
        __builtin_amdgcn_s_sleep(1);
        face_load(s0, fc);
      } while (missing());
    }
    face[0][lane] = fc.ny ? SfBits<T>::value(fc.y) : T(0);
    face[1][lane] = fc.nz ? SfBits<T>::value(fc.z) : T(0);
    __syncthreads(); // (one wavefront: orders the LDS accesses)
    T ey[C], ez[C];
#pragma unroll
    for (int j = 0; j < C; ++j) {
      ey[j] = face_y[j * kPen];
      ez[j] = face_z[j * kPen];
    }
    face_load(min(s0 + C, S - C), fc);
    const long u = (long)step(s0) * kWave, un = (long)step(ahead) * kWave;
    const int x0 = step(s0) - yl - zl, xn = step(ahead) - yl - zl;
#pragma unroll
    for (int j = 0; j < C; ++j) {
      const int x = UP ? x0 - j : x0 + j, q = j * dir;
      // The step's chain: a lane exchange, then a subtraction per neighbour. While the exchange is under way
      // the operands of a step of the next chunk are asked for.
      const T lz = UP ? __shfl_down(own, kPen, kWave) : __shfl_up(own, kPen, kWave);
      const T ly = lane_y<UP>(own);
      fetch(un, xn, j, o_next);
      const bool hasx = UP ? x < g.nx - 1 : x > 0;
      const T qy = face_lane_y ? ey[j] : ly, qx = hasx ? own : T(0);
      __builtin_amdgcn_sched_barrier(0);
      const T qz = face_lane_z ? ez[j] : lz;
      T v;
      // An absent neighbour's coefficient is +0 and so is its value here: subtracting their product changes
      // nothing, not even a zero's sign.
      if constexpr (KIND == kPenLower) {
        v = o.r[j] - o.z[j] * qz;
        v = v - o.y[j] * qy;
        v = v - o.x[j] * qx;
        (tt + u + lane)[q] = v;
      } else if constexpr (UP) {
        v = o.r[j] - o.x[j] * qx;
        v = v - o.y[j] * qy;
        v = v - o.z[j] * qz;
        v = v / o.d[j];
      } else {
        const T fz = hasz ? o.z[j] / qz : T(0), fy = hasy ? o.y[j] / qy : T(0), fx = hasx ? o.x[j] / own : T(0);
        v = o.d[j];
        if (hasz) v = v - fz * o.tz[j];
        if (hasy) v = v - fy * o.ty[j];
        if (hasx) v = v - fx * o.tx[j];
        (az + u + lane)[q] = fz;
        (ay + u + lane)[q] = fy;
        (ax + u + lane)[q] = fx;
        (dd + u + lane)[q] = v;
      }
      own = v;
      val[j][lane] = v;
    }
    __syncthreads();
    // (steps outside a line leave values there that nothing reads)
    const U vy = SfBits<T>::bits(val[fj][fk * kPen + far]), vz = SfBits<T>::bits(val[fj][far * kPen + fk]);
    const unsigned fo = (unsigned)step(s0 + fj) * kPen + fk;
    if (toy) __hip_atomic_store(yto + fo, vy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (toz) __hip_atomic_store(zto + fo, vz, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if constexpr (UP) {
      // the chunk's results, 8 consecutive x of 8 lines a store (a lane's own step by step is 64 lines a store):
      // step fk of the lines (fj, 0 .. 7)
      const int xs = step(s0 + fk) - fj, xend = b * kPen + fj < g.ny ? g.nx : 0;
      T* to = out + (((long)c * kPen * g.ny + b * kPen + fj) * g.nx + xs);
      T* none = tt + (long)(S - 1) * kWave; // a padding step's t is never read
#pragma unroll
      for (int m = 0; m < kPen; ++m) {
        const bool ok = (unsigned)(xs - m) < (unsigned)(c * kPen + m < g.nz ? xend : 0);
        *(ok ? to : none) = val[fk][m * kPen + fj];
        to += (long)g.ny * g.nx - 1;
      }
    }
    __syncthreads();
  };

  // two sets of operands in turn: the chunk's are used where they were loaded, no register is moved
  // (a copy would wait for its load)
  Ops even, odd;
#pragma unroll
  for (int j = 0; j < C; ++j) fetch((long)step(0) * kWave, step(0) - yl - zl, j, even);
  face_load(0, fc);
  for (int s0 = 0; s0 < S; s0 += 2 * C) {
    march(s0, even, min(s0 + C, S - C), odd);
    if (s0 + C >= S) break;
    march(s0 + C, odd, min(s0 + 2 * C, S - C), even);
  }
}

// A sweep pair (or a factorisation) with a wait that ran out of polls, again, by one workgroup and
// plane by plane of x + y + z, from the sweep that gave up; then the flags are cleared. Without a flag it returns at once.
constexpr int kPenRedoBlock = 1024;
template <typename T, bool FAC>
__global__ void __launch_bounds__(kPenRedoBlock) k_pencil_redo(PencilFactor<T> F, const double* trans, const T* in,
                                                                T* out, const int* __restrict__ done) {
  if (done && *done) return;
  const bool lower = __hip_atomic_load(F.work + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  if (!lower && __hip_atomic_load(F.work + 3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) return;
  const PencilGrid& g = F.g;
  const long np = g.positions();
  const int planes = g.nx + g.ny + g.nz - 2, lines = g.ny * g.nz;
  T *az = F.base, *ay = az + np, *ax = ay + np, *dd = ax + np, *ux = dd + np, *uy = ux + np, *uz = uy + np;
  auto each = [&](int d, auto f) {
    for (int l = threadIdx.x; l < lines; l += kPenRedoBlock) {
      const int y = l % g.ny, z = l / g.ny, x = d - y - z;
      if (x >= 0 && x < g.nx) f(x, y, z, g.position(x, y, z));
    }
    __syncthreads();
  };
  for (int d = 0; lower && d < planes; ++d)
    each(d, [&](int x, int y, int z, long q) {
      const T* from = FAC ? dd : F.t;
      const T vz = z > 0 ? from[g.position(x, y, z - 1)] : T(0), vy = y > 0 ? from[g.position(x, y - 1, z)] : T(0),
              vx = x > 0 ? from[g.position(x - 1, y, z)] : T(0);
      if (FAC) {
        T v = dd[q];
        if (z > 0) az[q] = az[q] / vz, v = v - az[q] * (T)trans[q];
        if (y > 0) ay[q] = ay[q] / vy, v = v - ay[q] * (T)trans[np + q];
        if (x > 0) ax[q] = ax[q] / vx, v = v - ax[q] * (T)trans[2 * np + q];
        dd[q] = v;
      } else {
        T v = in[((long)z * g.ny + y) * g.nx + x];
        if (z > 0) v = v - az[q] * vz;
        if (y > 0) v = v - ay[q] * vy;
        if (x > 0) v = v - ax[q] * vx;
        F.t[q] = v;
      }
    });
  if (!FAC)
    for (int d = planes - 1; d >= 0; --d)
      each(d, [&](int x, int y, int z, long q) {
        const long i = ((long)z * g.ny + y) * g.nx + x;
        T v = F.t[q];
        if (x < g.nx - 1) v = v - ux[q] * out[i + 1];
        if (y < g.ny - 1) v = v - uy[q] * out[i + g.nx];
        if (z < g.nz - 1) v = v - uz[q] * out[i + (long)g.nx * g.ny];
        out[i] = v / dd[q];
      });
  if (threadIdx.x < 2) __hip_atomic_store(F.work + 2 + threadIdx.x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

void launch_pencil_check(hipStream_t st, int n, const PencilGrid& g, const int* ro, const int* cols, int* bad) {
  hipLaunchKernelGGL(k_pencil_check, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, n, g, ro, cols, bad);
}

template <typename T>
void launch_pencil_init(hipStream_t st, const PencilFactor<T>& F) {
  const long nh = 2 * F.g.halo();
  hipLaunchKernelGGL(k_pencil_init<T>, dim3(grid_for(nh, 4)), dim3(kBlock), 0, st, nh, F.halo, F.work);
}

void launch_pencil_factor(hipStream_t st, const PencilFactor<double>& F, const int* ro, const double* vals,
                          double* trans, bool redo) {
  hipLaunchKernelGGL(k_pencil_fill, dim3((unsigned)((F.g.positions() + kBlock - 1) / kBlock)), dim3(kBlock), 0, st,
                     F.g, ro, vals, F.base, trans);
  if (redo)
    hipLaunchKernelGGL((k_pencil_redo<double, true>), dim3(1), dim3(kPenRedoBlock), 0, st, F, (const double*)trans,
                       (const double*)nullptr, (double*)nullptr, (const int*)nullptr);
  else
    hipLaunchKernelGGL((k_pencil_sweep<double, kPenFactor>), dim3(F.g.pencils()), dim3(kWave), 0, st, F,
                       (const double*)trans, (const double*)nullptr, (double*)nullptr, g_ilu_sf_spins,
                       (const int*)nullptr);
}

void launch_pencil_demote(hipStream_t st, const PencilFactor<double>& F, float* base) {
  const long n = 7 * F.g.positions();
  hipLaunchKernelGGL(k_pencil_demote, dim3(grid_for(n, 4)), dim3(kBlock), 0, st, n, (const double*)F.base, base);
}

void launch_pencil_to_csr(hipStream_t st, int n, const PencilFactor<double>& F, const int* ro, double* lu) {
  hipLaunchKernelGGL(k_pencil_to_csr, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, n, F.g, ro,
                     (const double*)F.base, lu);
}

template <typename T>
void launch_pencil_apply(hipStream_t st, const PencilFactor<T>& F, const T* y, T* x, const int* done) {
  const dim3 grid(F.g.pencils()), blk(kWave);
  const double* none = nullptr;
  hipLaunchKernelGGL((k_pencil_sweep<T, kPenLower>), grid, blk, 0, st, F, none, y, x, g_ilu_sf_spins, done);
  hipLaunchKernelGGL((k_pencil_sweep<T, kPenUpper>), grid, blk, 0, st, F, none, y, x, g_ilu_sf_spins, done);
  hipLaunchKernelGGL((k_pencil_redo<T, false>), dim3(1), dim3(kPenRedoBlock), 0, st, F, none, y, x, done);
}

template void launch_pencil_init<double>(hipStream_t, const PencilFactor<double>&);
template void launch_pencil_init<float>(hipStream_t, const PencilFactor<float>&);
template void launch_pencil_apply<double>(hipStream_t, const PencilFactor<double>&, const double*, double*, const int*);
template void launch_pencil_apply<float>(hipStream_t, const PencilFactor<float>&, const float*, float*, const int*);

} // namespace alien_hip
