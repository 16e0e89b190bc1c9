// HIP execution context of the backend: one stream, the workspace of the
// one-pass reductions, a ring of device-resident scalar slots and the pinned
// words through which scalars reach the host. Plays the part of the SYCL queue
// holder of Alien's SYCL backend (sycl/algebra/SYCLKernelInternal.h:32-84).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstddef>
#include <map>
#include <mutex>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "../../kernels/device_common.h"
#include "../../kernels/krylov_state.h"
#include "../../kernels/launch.h"

namespace alien_hip {

struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define ALIEN_HIP_CHECK(expr)                                                                 \
  do {                                                                                        \
    hipError_t _e = (expr);                                                                   \
    if (_e != hipSuccess)                                                                     \
      throw ::alien_hip::Error((int)_e, std::string(#expr) + ": " + hipGetErrorString(_e));   \
  } while (0)

// Check of the most recent launch(es) on this thread.
inline void check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) throw Error((int)e, std::string(what) + ": " + hipGetErrorString(e));
}

// Freed device blocks of 1 MiB or more, kept by device and size for the next allocation of that
// size: the solvers' work vectors are created and destroyed with each solve, and mapping and
// unmapping device memory each time costs milliseconds. A block is kept only after a device-wide
// synchronisation (what hipFree does), so no queued work can still use it when it is handed out
// again; at most 16 GiB are kept per process, and a failed hipMalloc empties the cache and tries
// once more. The cache is never destroyed (blocks are released with the process).
class BlockCache {
 public:
  static BlockCache& get() {
    static BlockCache* c = new BlockCache();
    return *c;
  }
  void* take(int dev, size_t bytes) {
    std::lock_guard<std::mutex> g(m_);
    auto it = free_.find({dev, bytes});
    if (it == free_.end() || it->second.empty()) return nullptr;
    void* p = it->second.back();
    it->second.pop_back();
    kept_ -= bytes;
    return p;
  }
  // true when the block was kept (else the caller frees it)
  bool give(int dev, void* p, size_t bytes) {
    if (bytes < kMin) return false;
    int cur = -1;
    if (hipGetDevice(&cur) != hipSuccess || cur != dev) return false;
    {
      std::lock_guard<std::mutex> g(m_);
      if (kept_ + bytes > kMax) return false;
    }
    if (hipDeviceSynchronize() != hipSuccess) return false;
    std::lock_guard<std::mutex> g(m_);
    if (kept_ + bytes > kMax) return false;
    free_[{dev, bytes}].push_back(p);
    kept_ += bytes;
    return true;
  }
  void release(int dev) {
    std::lock_guard<std::mutex> g(m_);
    for (auto& e : free_)
      if (e.first.first == dev) {
        for (void* p : e.second) {
          (void)hipFree(p);
          kept_ -= e.first.second;
        }
        e.second.clear();
      }
  }

 private:
  static constexpr size_t kMin = size_t(1) << 20, kMax = size_t(16) << 30;
  std::mutex m_;
  std::map<std::pair<int, size_t>, std::vector<void*>> free_;
  size_t kept_ = 0;
};

// Owning device array (its blocks of 1 MiB or more go through BlockCache).
template <typename T>
class DeviceArray {
 public:
  DeviceArray() = default;
  explicit DeviceArray(size_t n) { resize(n); }
  ~DeviceArray() { reset(); }
  DeviceArray(const DeviceArray&) = delete;
  DeviceArray& operator=(const DeviceArray&) = delete;
  DeviceArray(DeviceArray&& o) noexcept : m_p(o.m_p), m_n(o.m_n), m_dev(o.m_dev) { o.m_p = nullptr; o.m_n = 0; }
  DeviceArray& operator=(DeviceArray&& o) noexcept {
    if (this != &o) { reset(); m_p = o.m_p; m_n = o.m_n; m_dev = o.m_dev; o.m_p = nullptr; o.m_n = 0; }
    return *this;
  }
  void resize(size_t n) {
    reset();
    if (n) {
      const size_t bytes = n * sizeof(T);
      ALIEN_HIP_CHECK(hipGetDevice(&m_dev));
      m_p = static_cast<T*>(BlockCache::get().take(m_dev, bytes));
      if (!m_p) {
        hipError_t e = hipMalloc((void**)&m_p, bytes);
        if (e == hipErrorOutOfMemory) {
          (void)hipGetLastError();
          BlockCache::get().release(m_dev);
          e = hipMalloc((void**)&m_p, bytes);
        }
        if (e != hipSuccess) {
          m_p = nullptr;
          ALIEN_HIP_CHECK(e);
        }
      }
    }
    m_n = n;
  }
  // The same for workspace that its user can do without: false, and empty, where there is no memory for it.
  bool try_resize(size_t n) {
    try {
      resize(n);
    } catch (const Error& e) {
      if (e.code != (int)hipErrorOutOfMemory) throw;
      (void)hipGetLastError();
      return false;
    }
    return true;
  }
  void reset() {
    if (m_p && !BlockCache::get().give(m_dev, m_p, m_n * sizeof(T))) (void)hipFree(m_p);
    m_p = nullptr;
    m_n = 0;
  }
  // Synchronous upload: the host buffer may be reused or freed on return.
  void upload(const T* host, size_t n, hipStream_t st) {
    if (n != m_n) resize(n);
    if (n) {
      ALIEN_HIP_CHECK(hipMemcpyAsync(m_p, host, n * sizeof(T), hipMemcpyHostToDevice, st));
      ALIEN_HIP_CHECK(hipStreamSynchronize(st));
    }
  }
  T* data() { return m_p; }
  const T* data() const { return m_p; }
  size_t size() const { return m_n; }
  bool empty() const { return m_n == 0; }

 private:
  T* m_p = nullptr;
  size_t m_n = 0;
  int m_dev = 0;
};

} // namespace alien_hip

// The context object handed through the C ABI.
struct alien_hip_ctx {
  hipStream_t stream = nullptr;
  bool own_stream = false;
  bool trace = false; // ALIEN_HIP_TRACE=1 at creation: set-up phase times and mixed BiCGStab updates on stderr
  // Step-kernel timing (alien_hip_ctx_step_timing): when on, the fused CG solvers bracket each
  // launch of their q = A p kernel with HIP events on `stream` and add up the durations here
  bool step_timing = false;
  double step_us = 0.0;
  long long step_launches = 0;
  // reduction workspace (see RedWork); grows on demand, never while a graph is captured
  alien_hip::DeviceArray<double> partials;
  int red_cap = 0;
  alien_hip::DeviceArray<double> scalars; // device-resident scalar slots
  // zeroed CG state (done = 0, never written): the fused iteration's kernels launched on their own
  alien_hip::DeviceArray<alien_hip::CGState> idle_cg;
  // slots and head of the grid-wide sums of the resident CG (cg_resident.hip), zeros at first
  alien_hip::DeviceArray<unsigned long long> grid_slots;
  alien_hip::DeviceArray<int> grid_head;
  // Zeros again, on the stream: after a launch that gave up, whose words are tagged with phases past the head's, which
  // the next launch would take for its own.
  void clear_grid() {
    ALIEN_HIP_CHECK(hipMemsetAsync(grid_slots.data(), 0, sizeof(unsigned long long) * grid_slots.size(), stream));
    ALIEN_HIP_CHECK(hipMemsetAsync(grid_head.data(), 0, sizeof(int) * grid_head.size(), stream));
  }
  // pivots (one per row, in the last block) and ticket, flag of the ILU(0) kernels of ilu0_sync.hip
  // Threads that call the entry points on one context take turns to queue a call's launches: the first of them clears
  // what the others use.
  std::mutex ilu_turn;
  std::vector<alien_hip::DeviceArray<double>> ilu_piv;
  alien_hip::DeviceArray<int> ilu_work;
  // Room for them, without a wait for the stream: a block that has become too small stays (queued launches may use it)
  // until the context goes, and each is at least twice the one before, so that all of them are at most twice the last.
  // False without the memory for it, and inside a stream capture: a graph would outlive the workspace, and its replays
  // beside the context's own work would share ticket, flag and pivots with it.
  bool reserve_ilu(size_t rows) {
    if (capturing()) return false;
    const size_t have = ilu_piv.empty() ? 0 : ilu_piv.back().size();
    if (have >= rows) return true;
    alien_hip::DeviceArray<double> more;
    if (!more.try_resize(std::max(rows, 2 * have))) return false;
    ilu_piv.push_back(std::move(more));
    return true;
  }
  bool capturing() const {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    ALIEN_HIP_CHECK(hipStreamIsCapturing(stream, &cap));
    return cap != hipStreamCaptureStatusNone;
  }
  int device = 0, cus = 0; // the context's device and its compute units
  // resident CG (cg_resident.hip): on / off (ALIEN_HIP_CG_RESIDENT at creation), polls of a wait
  // before it gives up (ALIEN_HIP_CG_RESIDENT_SPINS)
  bool cg_resident = true;
  long resident_spins = 1L << 20;
  // pinned, coherent words that kernels post to (HostPost): two for each scalar slot, then a state's
  unsigned long long* mail = nullptr;
  static constexpr int kMailWords = 2 * 64 + alien_hip::kMaxPostWords;
  unsigned last_tag = 0, slot_tag[64] = {}; // tag of the post that fills a slot's words (0: none under way)
  unsigned waits = 0;
  double poll_s = 4e-3; // a read polls its posted words as long before it waits for the stream; 0: the program asked for blocking waits
  alien_hip::DeviceArray<unsigned> tickets; // counters of the reductions finished in their own launch, zeros
  // Pinned 512-byte blocks for the fused solvers' host state mirrors, allocated once per context
  // (pinned allocation and release cost far more than a solve's own host work); a solver takes a
  // free block and gives it back, or allocates its own when all are taken.
  static constexpr int kPinnedBlocks = 16, kPinnedBytes = 512;
  char* pinned_blocks = nullptr;
  unsigned pinned_used = 0;
  void* take_pinned() {
    if (!pinned_blocks &&
        hipHostMalloc((void**)&pinned_blocks, (size_t)kPinnedBlocks * kPinnedBytes, hipHostMallocDefault) != hipSuccess) {
      pinned_blocks = nullptr;
      return nullptr;
    }
    for (int i = 0; i < kPinnedBlocks; ++i)
      if (!(pinned_used & (1u << i))) {
        pinned_used |= 1u << i;
        return pinned_blocks + (size_t)i * kPinnedBytes;
      }
    return nullptr;
  }
  // false when p is not one of the blocks (the caller frees it)
  bool give_pinned(void* p) {
    if (!pinned_blocks || (char*)p < pinned_blocks || (char*)p >= pinned_blocks + kPinnedBlocks * kPinnedBytes)
      return false;
    pinned_used &= ~(1u << (int)(((char*)p - pinned_blocks) / kPinnedBytes));
    return true;
  }
  int next_slot = 0;
  static constexpr int kSlots = 64;

  // Make room for reductions launched with up to `nblocks` workgroups.
  void reserve_red(long nblocks) {
    if (nblocks <= red_cap) return;
    long cap = red_cap ? red_cap : 4096;
    while (cap < nblocks) cap *= 2;
    ALIEN_HIP_CHECK(hipStreamSynchronize(stream));
    partials.resize((size_t)alien_hip::kMaxSlots * cap);
    red_cap = (int)cap;
  }
  // Room for every kernel of this library on vectors of n rows.
  void reserve_for(long n) {
    long b = alien_hip::bundle_blocks_max(n);
    long e = alien_hip::ept_blocks(n);
    long r = (n + alien_hip::kBlock - 1) / alien_hip::kBlock;
    reserve_red(std::max(b, std::max(e, r)));
  }
  alien_hip::RedWork red() {
    return alien_hip::RedWork{partials.data(), red_cap};
  }
  // The same for a reduction that may finish in its own launch: not inside a stream capture, since a graph
  // replayed beside the context's own work would leave the counters wrong for good, not for one result.
  alien_hip::RedWork red_once() {
    alien_hip::RedWork w = red();
    if (!capturing()) w.ticket = tickets.data();
    return w;
  }
  // A fresh device scalar slot (ring of kSlots; callers keep at most a few live).
  int take_slot() {
    int s = next_slot;
    next_slot = (next_slot + 1) % kSlots;
    slot_tag[s] = 0;
    return s;
  }
  double* dslot(int s) { return scalars.data() + s; }
  // Where the kernel that writes slot s posts it too, for a read_slot that follows at once. (Nothing that a stream
  // capture may record posts by itself: each replay would post under the same tag, and a read would take the first
  // replay's value for the last one's.)
  alien_hip::HostPost post_slot(int s) {
    slot_tag[s] = new_tag();
    return alien_hip::HostPost{mail + 2 * s, slot_tag[s]};
  }
  // One slot's value once the work queued before has written it.
  double read_slot(int s) {
    double v;
    if (!slot_tag[s]) alien_hip::launch_post_words(stream, dslot(s), 2, post_slot(s));
    const unsigned tag = slot_tag[s];
    slot_tag[s] = 0;
    fetch(mail + 2 * s, tag, dslot(s), &v, 2);
    return v;
  }
  // The same in two halves: the words asked for (one such question at a time); looked at; waited for.
  alien_hip::HostPost ask_words(const void* from, int n) {
    const alien_hip::HostPost p{mail + 2 * kSlots, new_tag()};
    alien_hip::launch_post_words(stream, from, n, p);
    return p;
  }
  bool peek_words(const alien_hip::HostPost& p, void* to, int n) const { return arrived(p.to, p.tag, static_cast<unsigned*>(to), n); }
  void take_words(const alien_hip::HostPost& p, const void* from, void* to, int n) { fetch(p.to, p.tag, from, to, n); }
  // n 32-bit words of device memory, likewise, and one from `also` (at most kMaxPostWords together).
  void read_words(const void* from, void* to, int n, const int* also = nullptr, int* also_to = nullptr) {
    const alien_hip::HostPost p{mail + 2 * kSlots, new_tag()};
    alien_hip::launch_post_words(stream, from, n, p, also);
    fetch(p.to, p.tag, from, to, n);
    if (also) fetch(p.to + n, p.tag, also, also_to, 1);
  }

 private:
  static bool arrived(const unsigned long long* from, unsigned tag, unsigned* out, int n) {
    for (int i = 0; i < n; ++i) {
      const unsigned long long w = __atomic_load_n(from + i, __ATOMIC_ACQUIRE);
      if ((unsigned)(w >> 32) != tag) return false;
      out[i] = (unsigned)w;
    }
    return true;
  }
  unsigned new_tag() { return last_tag += last_tag == ~0u ? 2 : 1; }
  // The words posted with this tag. The host polls memory: a stored word reaches it in about 2 us, where a
  // copy and a wait for the stream took 13 to 20. After 4 ms, where those no longer matter, it waits for the
  // stream and leaves its core to others. A word that the finished stream has not posted is copied.
  void fetch(const unsigned long long* from, unsigned tag, const void* dev, void* to, int n) {
    alien_hip::check_launch("post");
    unsigned* out = static_cast<unsigned*>(to);
    const auto now = std::chrono::steady_clock::now;
    const auto until = now() + std::chrono::duration<double>(poll_s);
    for (unsigned spin = 1; !arrived(from, tag, out, n); ++spin) {
      if (poll_s > 0 && (spin % 64 || now() < until)) {
        __builtin_ia32_pause();
        continue;
      }
      ALIEN_HIP_CHECK(hipStreamSynchronize(stream));
      if (arrived(from, tag, out, n)) break;
      ALIEN_HIP_CHECK(hipMemcpyAsync(to, dev, sizeof(unsigned) * n, hipMemcpyDeviceToHost, stream));
      ALIEN_HIP_CHECK(hipStreamSynchronize(stream));
      return;
    }
    // the runtime frees what it keeps of finished launches when it is asked to wait
    if (++waits % 256 == 0) ALIEN_HIP_CHECK(hipStreamSynchronize(stream));
  }
};

namespace alien_hip {
alien_hip_ctx* default_ctx();
alien_hip_ctx* make_ctx(void* stream);
void destroy_ctx(alien_hip_ctx* c);
} // namespace alien_hip
