// What calls leave in the state of a context: calls off the straight path (a wait given up, a stream capture, a second
// context, a result in its operand's place, a device without memory), followed by ordinary ones on the same context.
// Prints one JSON object per check on stdout for tests/test_gpu_ctx_state.py. The internal headers give the checks the
// context's own fields.
// Usage: ctx_state_check [check ...]  (all of them without an argument; blocking_wait has to come first)
#include <dlfcn.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <ctime>
#include <functional>
#include <map>
#include <random>
#include <string>
#include <vector>

#include "alien/hip/HIPBackEnd.h"
#include "alien/hip/krylov/HIPILU0Preconditioner.h"
#include "kernels/resident_turn.h"

// Device allocations of `refuse` bytes end as those of a device without memory (this definition comes before the runtime's).
static size_t refuse = 0;
static int refused = 0;
extern "C" hipError_t hipMalloc(void** p, size_t bytes) {
  typedef hipError_t (*Malloc)(void**, size_t);
  static const Malloc real = (Malloc)dlsym(RTLD_NEXT, "hipMalloc");
  if (bytes != refuse || bytes == 0) return real(p, bytes);
  ++refused;
  return real(p, size_t(1) << 46);
}

namespace {

struct System {
  int n = 0;
  std::vector<int> ro, cols;
  std::vector<double> vals, b;
};

// 7-point system, its right-hand side the product with U[0,1) values of `seed`
System generate(int kind, int nx, int ny, int nz, unsigned seed) {
  System a;
  const long nnz = alien_hip_gen_nnz(kind, nx, ny, nz);
  a.n = nx * ny * nz;
  a.ro.resize(a.n + 1);
  a.cols.resize(nnz);
  a.vals.resize(nnz);
  const double lognormal[4] = {1, 1, 1, 1};
  if (alien_hip_gen_csr(kind, nx, ny, nz, kind == ALIEN_HIP_GEN_LOGNORMAL7 ? lognormal : nullptr, seed, a.ro.data(),
                        a.cols.data(), a.vals.data()) != 0) {
    std::fprintf(stderr, "gen_csr: %s\n", alien_hip_last_error());
    std::exit(2);
  }
  std::vector<double> x(a.n);
  alien_hip_fill_uniform01(seed, a.n, x.data());
  a.b.assign(a.n, 0);
  for (int i = 0; i < a.n; ++i)
    for (int k = a.ro[i]; k < a.ro[i + 1]; ++k) a.b[i] += a.vals[k] * x[a.cols[k]];
  return a;
}

void call(int rc, const char* what) {
  if (rc == 0) return;
  std::fprintf(stderr, "%s: %s\n", what, alien_hip_last_error());
  std::exit(3);
}

struct Context {
  alien_hip_ctx* c = nullptr;
  Context() { call(alien_hip_ctx_create(nullptr, &c), "ctx_create"); }
  ~Context() { alien_hip_ctx_destroy(c); }
  alien_hip_ctx* operator->() const { return c; }
};

struct Solved {
  std::vector<double> x;
  alien_hip_solve_result r{};
  bool operator==(const Solved& o) const {
    return r.iterations == o.r.iterations && r.status == o.r.status && r.error == o.r.error &&
           std::memcmp(x.data(), o.x.data(), sizeof(double) * x.size()) == 0;
  }
};

alien_hip_solve_params params(int precond, int mode, double tol) {
  alien_hip_solve_params p{};
  p.solver = ALIEN_HIP_CG;
  p.precond = precond;
  p.layout = ALIEN_HIP_LAYOUT_RBDIA;
  p.mode = mode;
  p.tol = tol;
  p.max_iter = 2000;
  p.poll_every = 8;
  return p;
}

Solved solve(const Context& c, const System& a, int mode, double tol = 1e-10, int precond = ALIEN_HIP_PREC_DIAG) {
  Solved s;
  s.x.assign(a.n, 0.0);
  const alien_hip_solve_params p = params(precond, mode, tol);
  call(alien_hip_solve_csr(c.c, &p, a.n, a.ro.data(), a.cols.data(), a.vals.data(), a.b.data(), s.x.data(), &s.r),
       "solve_csr");
  return s;
}

template <typename T>
std::vector<T> read(const alien_hip::DeviceArray<T>& d) {
  std::vector<T> h(d.size());
  ALIEN_HIP_CHECK(hipDeviceSynchronize());
  ALIEN_HIP_CHECK(hipMemcpy(h.data(), d.data(), sizeof(T) * h.size(), hipMemcpyDeviceToHost));
  return h;
}

// After waits given up, the words of the grid-wide sums hold no phase that a later launch will reach, and solves of other
// systems with the usual number of polls are those of a context that runs no resident launch.
void after_a_wait_given_up() {
  const System first = generate(ALIEN_HIP_GEN_LOGNORMAL7, 40, 41, 43, 1);
  const System second = generate(ALIEN_HIP_GEN_LOGNORMAL7, 44, 37, 45, 2);
  Context launches, c;
  launches->cg_resident = false;
  const long usual = c->resident_spins;
  int newer = 0, gave_up = 1, same = 1;
  for (int mode : {ALIEN_HIP_MODE_GRAPH, ALIEN_HIP_MODE_MIXED}) {
    c->resident_spins = 0;
    gave_up &= solve(c, first, mode).r.status;
    const unsigned head = (unsigned)read(c->grid_head)[0];
    for (unsigned long long w : read(c->grid_slots)) newer += (unsigned)(w >> 32) > head;
    c->resident_spins = usual;
    same &= solve(c, second, mode) == solve(launches, second, mode);
  }
  std::printf("{\"check\": \"after_a_wait_given_up\", \"status\": %d, \"newer_words\": %d, \"same\": %d}\n", gave_up, newer,
              same);
}

// With the flag of a wait given up raised, whatever the launch's own state says: the solve goes on from the true residual
// and the flag is down again.
void flag_is_read() {
  const System a = generate(ALIEN_HIP_GEN_LOGNORMAL7, 40, 41, 43, 3);
  const double tol = 1e-10;
  Context c;
  int up = 0, status = 1;
  double worst = 0;
  for (int mode : {ALIEN_HIP_MODE_GRAPH, ALIEN_HIP_MODE_MIXED}) {
    const int one = 1;
    ALIEN_HIP_CHECK(hipMemcpy(c->grid_head.data() + 1, &one, sizeof(int), hipMemcpyHostToDevice));
    const Solved s = solve(c, a, mode, tol);
    status &= s.r.status;
    worst = std::max(worst, s.r.true_rel_res / tol);
    up += read(c->grid_head)[1];
  }
  std::printf("{\"check\": \"flag_is_read\", \"status\": %d, \"up\": %d, \"residual\": %.17g}\n", status, up, worst);
}

// A kept matrix solved through another context than the one it was made on leaves that one's scalar slots alone (another
// thread may be solving there), with the same result.
void matrix_of_another_context() {
  const System a = generate(ALIEN_HIP_GEN_LOGNORMAL7, 81, 81, 81, 4);
  Context own, other;
  Solved got[2];
  int moved = 0;
  for (const Context* c : {&other, &own}) {
    alien_hip_matrix* m = nullptr;
    call(alien_hip_matrix_create(own.c, a.n, a.ro.data(), a.cols.data(), a.vals.data(), &m), "matrix_create");
    const int slot = own->next_slot;
    Solved& s = got[c == &own];
    s.x.assign(a.n, 0.0);
    alien_hip_solve_params p = params(ALIEN_HIP_PREC_DIAG, ALIEN_HIP_MODE_MIXED, 1e-8);
    p.max_iter = 40;
    call(alien_hip_solve(c->c, &p, m, a.b.data(), s.x.data(), &s.r), "solve");
    if (c == &other) moved = own->next_slot != slot;
    alien_hip_matrix_destroy(m);
  }
  std::printf("{\"check\": \"matrix_of_another_context\", \"moved\": %d, \"same\": %d}\n", moved, got[0] == got[1]);
}

// A dot product into a future, captured: the future gives the last replay's value, not the first one's.
void captured_dot() {
  Context c;
  const int n = 5000;
  Alien::HIPInternalLinearAlgebra alg(c.c);
  Alien::HIPVector x(Alien::HIPResource{n, c.c});
  const std::vector<double> ones(n, 1.0);
  x.setValues(ones.data());
  double v = 0;
  Alien::HIPFuture f(v);
  hipGraph_t g;
  hipGraphExec_t e;
  ALIEN_HIP_CHECK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  alg.dot(x, x, f);
  ALIEN_HIP_CHECK(hipStreamEndCapture(c->stream, &g));
  ALIEN_HIP_CHECK(hipGraphInstantiate(&e, g, nullptr, nullptr, 0));
  for (int k = 1; k <= 3; ++k) {
    const std::vector<double> h(n, (double)k);
    x.setValues(h.data());
    ALIEN_HIP_CHECK(hipGraphLaunch(e, c->stream));
    ALIEN_HIP_CHECK(hipStreamSynchronize(c->stream));
  }
  const double got = f.get(), eager = alg.dot(x, x);
  ALIEN_HIP_CHECK(hipGraphExecDestroy(e));
  ALIEN_HIP_CHECK(hipGraphDestroy(g));
  std::printf("{\"check\": \"captured_dot\", \"value\": %.17g, \"eager\": %.17g}\n", got, eager);
}

// A future's get() returns when what was queued behind the dot is done too. (An event tells: the stream itself may not yet
// be idle, the launch that handed the value over being its last.)
void future_synchronises() {
  Context c;
  const int n = 5000;
  Alien::HIPInternalLinearAlgebra alg(c.c);
  Alien::HIPVector x(Alien::HIPResource{n, c.c});
  const std::vector<double> ones(n, 1.0);
  x.setValues(ones.data());
  const size_t bytes = size_t(1) << 30;
  alien_hip::DeviceArray<char> a(bytes), b(bytes);
  double v = 0;
  Alien::HIPFuture f(v);
  alg.dot(x, x, f);
  for (int k = 0; k < 100; ++k)  // 40 ms
    ALIEN_HIP_CHECK(hipMemcpyAsync(a.data(), b.data(), bytes, hipMemcpyDeviceToDevice, c->stream));
  hipEvent_t copied;
  ALIEN_HIP_CHECK(hipEventCreate(&copied));
  ALIEN_HIP_CHECK(hipEventRecord(copied, c->stream));
  const double got = f.get();
  const bool done = hipEventQuery(copied) == hipSuccess;
  ALIEN_HIP_CHECK(hipEventDestroy(copied));
  std::printf("{\"check\": \"future_synchronises\", \"value\": %.17g, \"done\": %d}\n", got, done);
}

// ILU(0) in pencils, the result in the right-hand side's place, with every wait given up and with none: as apart.
void pencils_in_place() {
  const System a = generate(ALIEN_HIP_GEN_CONVDIFF7, 21, 18, 19, 5);
  Context c;
  Alien::HIPInternalLinearAlgebra alg(c.c);
  Alien::HIPMatrix A(static_cast<const Alien::MultiMatrixImpl*>(nullptr));
  A.build(c.c, Alien::CSRHostView{a.n, a.ro.data(), a.cols.data(), a.vals.data()}, Alien::kLayoutCSR);
  const long usual = alien_hip::g_ilu_sf_spins;
  std::vector<double> x[3];
  bool pencils = true;
  for (int k = 0; k < 3; ++k) { // apart; in place; in place, given up
    alien_hip::g_ilu_sf_spins = usual;
    Alien::ILU0Preconditioner<Alien::HIPInternalLinearAlgebra> P(alg, A);
    P.init();
    pencils = pencils && P.pencils();
    Alien::HIPVector y(A.resource()), z(A.resource());
    y.setValues(a.b.data());
    alien_hip::g_ilu_sf_spins = k == 2 ? 0 : usual;
    P.solve(alg, y, k == 0 ? z : y);
    x[k].resize(a.n);
    (k == 0 ? z : y).copyValuesTo(x[k].data());
  }
  alien_hip::g_ilu_sf_spins = usual;
  std::printf("{\"check\": \"pencils_in_place\", \"pencils\": %d, \"in_place\": %d, \"given_up\": %d}\n", pencils,
              x[1] == x[0], x[2] == x[0]);
}

// init() again with a colour schedule and new values on a preconditioner that had taken pencils: the new factor's sweeps.
void colours_after_pencils() {
  const System a = generate(ALIEN_HIP_GEN_CONVDIFF7, 10, 8, 8, 6);
  Context c;
  Alien::HIPInternalLinearAlgebra alg(c.c);
  Alien::HIPMatrix A(static_cast<const Alien::MultiMatrixImpl*>(nullptr));
  A.build(c.c, Alien::CSRHostView{a.n, a.ro.data(), a.cols.data(), a.vals.data()}, Alien::kLayoutCSR);
  Alien::ILU0Preconditioner<Alien::HIPInternalLinearAlgebra> P(alg, A), fresh(alg, A);
  P.init();
  const bool pencils = P.pencils();
  std::vector<double> vals(a.vals), x[2];
  for (size_t k = 0; k < vals.size(); ++k) vals[k] *= 1.0 + 0.01 * (k % 7);
  A.updateValues(vals.data());
  std::vector<int> colours(a.n + 1); // each row a colour of its own
  for (int i = 0; i <= a.n; ++i) colours[i] = i;
  P.setColourSchedule(colours);
  P.init();
  fresh.init();
  Alien::HIPVector y(A.resource()), z(A.resource());
  y.setValues(a.b.data());
  for (int k = 0; k < 2; ++k) {
    (k == 0 ? P : fresh).solve(alg, y, z);
    x[k].resize(a.n);
    z.copyValuesTo(x[k].data());
  }
  std::printf("{\"check\": \"colours_after_pencils\", \"pencils\": [%d, %d], \"same\": %d}\n", pencils, P.pencils(),
              x[0] == x[1]);
}

// Solves of one workgroup go on while another launch holds every compute unit, of a few workgroups while the others are held.
void small_solves_take_their_share() {
  const System one = generate(ALIEN_HIP_GEN_LOGNORMAL7, 14, 11, 9, 7), few = generate(ALIEN_HIP_GEN_LOGNORMAL7, 21, 18, 19, 8);
  Context c;
  int status = 0;
  {
    const alien_hip::ResidentTurn all(alien_hip::resident_gate(c->device), c->cus, c->cus);
    status += solve(c, one, ALIEN_HIP_MODE_GRAPH).r.status;
  }
  const alien_hip::ResidentTurn rest(alien_hip::resident_gate(c->device), c->cus - 8, c->cus);
  status += solve(c, few, ALIEN_HIP_MODE_GRAPH).r.status;
  std::printf("{\"check\": \"small_solves_take_their_share\", \"solved\": %d}\n", status);
}

// A program that asked for blocking waits (before anything else on the device) gets them from a read-back too.
void blocking_wait() {
  ALIEN_HIP_CHECK(hipSetDeviceFlags(hipDeviceScheduleBlockingSync));
  Context c;
  const int n = 5000;
  Alien::HIPInternalLinearAlgebra alg(c.c);
  Alien::HIPVector x(Alien::HIPResource{n, c.c});
  const std::vector<double> ones(n, 1.0);
  x.setValues(ones.data());
  const size_t bytes = size_t(1) << 30;
  alien_hip::DeviceArray<char> a(bytes), b(bytes);
  double v = alg.dot(x, x);
  for (int k = 0; k < 200; ++k)  // 90 ms
    ALIEN_HIP_CHECK(hipMemcpyAsync(a.data(), b.data(), bytes, hipMemcpyDeviceToDevice, c->stream));
  auto now = [](clockid_t id) {
    timespec t;
    clock_gettime(id, &t);
    return t.tv_sec + 1e-9 * t.tv_nsec;
  };
  const double wall = now(CLOCK_MONOTONIC), cpu = now(CLOCK_THREAD_CPUTIME_ID);
  v = alg.dot(x, x);
  std::printf("{\"check\": \"blocking_wait\", \"value\": %.17g, \"wall_s\": %.4f, \"cpu_s\": %.4f}\n", v,
              now(CLOCK_MONOTONIC) - wall, now(CLOCK_THREAD_CPUTIME_ID) - cpu);
}

// Which rows' systems run in one launch: the phase in the context's head tells. Rows of 6 to 9 entries, in one workgroup and
// in several.
void widths_in_one_launch() {
  std::printf("{\"check\": \"widths_in_one_launch\", \"taken\": [");
  for (int width = 6; width <= 9; ++width)
    for (int n : {1000, 5000}) {
      System a;
      a.n = n;
      a.ro.push_back(0);
      a.b.assign(n, 1.0);
      const std::vector<int> offsets = {0, -1, 1, -5, 5, -37, 37, -41, 41};
      for (int i = 0; i < n; ++i) {
        std::vector<int> c;
        for (int k = 0; k < width; ++k)
          if (i + offsets[k] >= 0 && i + offsets[k] < n) c.push_back(i + offsets[k]);
        std::sort(c.begin(), c.end());
        for (int j : c) {
          a.cols.push_back(j);
          a.vals.push_back(j == i ? 9.0 : -1.0);
        }
        a.ro.push_back((int)a.cols.size());
      }
      Context c;
      solve(c, a, ALIEN_HIP_MODE_GRAPH);
      std::printf("%s%d", width == 6 && n == 1000 ? "" : ", ", read(c->grid_head)[0] != 0);
    }
  std::printf("]}\n");
}

// Without the memory for a faster form's workspace, calls run in the form that needs none, to the same bits.
void without_memory() {
  int failed = 0, same = 1;
  auto without = [&](size_t bytes, auto f) {
    refuse = bytes;
    refused = 0;
    auto r = f();
    failed += refused > 0;
    refuse = 0;
    return r;
  };
  const System a = generate(ALIEN_HIP_GEN_CONVDIFF7, 21, 18, 19, 9), s = generate(ALIEN_HIP_GEN_LOGNORMAL7, 21, 18, 19, 9);
  { // the ILU(0) entry points' pivots
    std::vector<int> dcol(a.n), level(a.n), rows(a.n);
    alien_hip::host_dcol(a.n, a.ro.data(), a.cols.data(), dcol.data());
    const int nl = alien_hip::host_levels(a.n, a.ro.data(), a.cols.data(), dcol.data(), 0, level.data());
    std::vector<int> ptr(nl + 1);
    alien_hip::group_by_level(a.n, level.data(), nl, ptr.data(), rows.data());
    auto factor = [&] {
      Context c;
      alien_hip::DeviceArray<int> ro, cols, d, r;
      alien_hip::DeviceArray<double> lu;
      ro.upload(a.ro.data(), a.ro.size(), c->stream);
      cols.upload(a.cols.data(), a.cols.size(), c->stream);
      d.upload(dcol.data(), dcol.size(), c->stream);
      r.upload(rows.data(), rows.size(), c->stream);
      lu.upload(a.vals.data(), a.vals.size(), c->stream);
      call(alien_hip_ilu0_factor_f64(c.c, a.n, ro.data(), cols.data(), d.data(), lu.data(), nl, ptr.data(), r.data()),
           "ilu0_factor");
      return read(lu);
    };
    same &= without(sizeof(double) * a.n, factor) == factor();
  }
  auto bicg = [&](int mode) {
    Context c;
    Solved r;
    r.x.assign(a.n, 0.0);
    alien_hip_solve_params p = params(ALIEN_HIP_PREC_ILU0, mode, 1e-10);
    p.solver = ALIEN_HIP_BICGS;
    call(alien_hip_solve_csr(c.c, &p, a.n, a.ro.data(), a.cols.data(), a.vals.data(), a.b.data(), r.x.data(), &r.r),
         "solve_csr");
    return r;
  };
  alien_hip::PencilGrid g;
  same &= alien_hip::pencil_grid(a.n, a.ro.data(), a.cols.data(), g);
  const size_t words = 8 * g.positions() + 2 * g.halo();
  same &= without(sizeof(double) * words, [&] { return bicg(ALIEN_HIP_MODE_GRAPH); }) == bicg(ALIEN_HIP_MODE_GRAPH);
  same &= without(sizeof(double) * 3 * g.positions(), [&] { return bicg(ALIEN_HIP_MODE_GRAPH); }) == bicg(ALIEN_HIP_MODE_GRAPH);
  same &= without(sizeof(float) * words, [&] { return bicg(ALIEN_HIP_MODE_MIXED); }) == bicg(ALIEN_HIP_MODE_MIXED);
  Context c; // the exchange vectors of CG in one launch
  same &= without(sizeof(double) * 2 * s.n, [&] { return solve(c, s, ALIEN_HIP_MODE_GRAPH); }) == solve(c, s, ALIEN_HIP_MODE_GRAPH);
  std::printf("{\"check\": \"without_memory\", \"refused\": %d, \"same\": %d}\n", failed, same);
}

const std::map<std::string, std::function<void()>> kChecks = {
    {"after_a_wait_given_up", after_a_wait_given_up},
    {"blocking_wait", blocking_wait},
    {"captured_dot", captured_dot},
    {"colours_after_pencils", colours_after_pencils},
    {"flag_is_read", flag_is_read},
    {"future_synchronises", future_synchronises},
    {"matrix_of_another_context", matrix_of_another_context},
    {"pencils_in_place", pencils_in_place},
    {"small_solves_take_their_share", small_solves_take_their_share},
    {"widths_in_one_launch", widths_in_one_launch},
    {"without_memory", without_memory},
};

} // namespace

int main(int argc, char** argv) {
  for (const auto& c : kChecks) {
    bool on = argc == 1;
    for (int k = 1; k < argc; ++k) on = on || c.first == argv[k];
    if (!on) continue;
    std::fprintf(stderr, "check %s\n", c.first.c_str());
    c.second();
    std::fflush(stdout);
  }
  return 0;
}
