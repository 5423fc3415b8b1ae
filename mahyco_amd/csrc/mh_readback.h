// mh_readback.h -- fields of the state to host memory.
//
// Two routes.  Plain: the runtime's copy into the caller's memory, and for values formed per cell from
// several arrays (a member environment's, the membership, Materiau) a loop over copies of those.
// Pinned: a kernel writes the field, or forms it, into a ring of pinned slots, which the calling thread
// and up to seven more empty.  (The copy engine takes longer into the same slots: 4 MB 595 us, 34 MB 1910.)
// One thread below 4 MB (two copy 1 MB no faster than one), one more per 2 MB, eight at most (12 are
// slower); 4 MB slots at most (57 MB with 2 MB ones: 3.8 ms instead of 3.4).
//
// Plain / pinned, us, one array into pages used before: 29 KB 34 / 35, 262 KB 41 / 45 (140 / 50 among a
// process's first reads), 1 MB 85 / 85, 2 MB 270 / 120, 4 MB 600 / 190, 8 MB 1200 / 255, 34 MB 5400 / 775;
// into new pages: 262 KB 85 / 85, 4 MB 1350 / 1000, 34 MB 12900 / 7500.  Formed values: 4.6 KB 60 / 32,
// 262 KB 85 / 43, 2 MB 960 / 115.  Pinning itself takes 0.1 ms for 64 KB and 1.3 ms from 2 MB on, once.  So
// one array below 64 KB always takes the plain route, and slots are pinned only when the reads since
// they were last given back would have gained by them what they cost: a case that reads one field of
// 2 MB takes 270 us for it, where pinning first took 1200.
//
// The slots belong to the process: at most two rings of 16 MB, each with one reader at a time (a read
// that finds none free takes the plain route), given back with the last case and ensemble.
#ifndef MH_READBACK_H
#define MH_READBACK_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "mh_math.h"
#include "mh_state.h"

// A ring of pinned slots.
struct HostStage {
  static constexpr int kSlots = 4;
  static constexpr size_t kArray = 64u << 10;  // one array: by the pinned route from here on
  char* pin = nullptr;
  size_t slot = 0;  // bytes of a slot
  int slots = 0;
  bool busy = false;  // a read uses it

  // the slots for n bytes: one that holds a small field; for larger ones a quarter each, as far as
  // 4 MB.  In powers of two, so that a node field after a cell field of the same mesh, or one case after
  // another, seldom asks for more
  static int count(size_t n) { return n <= (256u << 10) ? 1 : kSlots; }
  static size_t size(size_t n) {
    size_t s = 64u << 10;
    while (s * count(n) < n && s < (4u << 20)) s *= 2;
    return s;
  }
  bool holds(size_t n) const { return pin && slots * slot >= count(n) * size(n); }

  hipError_t reserve(size_t n) {
    if (holds(n)) return hipSuccess;
    release();
    hipError_t e = hipErrorOutOfMemory;
    for (size_t s = size(n); s >= (64u << 10); s /= 2) {  // with less where pinned memory is short
      e = hipHostMalloc((void**)&pin, count(n) * s, hipHostMallocPortable);  // for every device
      if (e == hipSuccess) {
        slot = s;
        slots = count(n);
        return e;
      }
      pin = nullptr;
      (void)hipGetLastError();
    }
    return e;
  }
  void release() {
    if (pin) (void)hipHostFree(pin);
    pin = nullptr;
    slot = 0;
    slots = 0;
  }
};

// The process's rings.
struct ReadPool {
  static constexpr int kRings = 2;
  std::mutex mu;
  HostStage ring[kRings];
  long users = 0;   // cases and ensembles alive
  double owed = 0.;  // us that the plain reads so far would have gained by the pinned route

  void enter() {
    std::lock_guard<std::mutex> lock(mu);
    ++users;
  }
  void leave() {
    std::lock_guard<std::mutex> lock(mu);
    if (--users) return;
    for (HostStage& r : ring) r.release();
    owed = 0.;
  }
  // A ring for a read of n bytes that gains `gain` us by it, or null where the plain route is taken.
  HostStage* take(size_t n, double gain) {
    std::lock_guard<std::mutex> lock(mu);
    HostStage* got = nullptr;
    for (HostStage& r : ring) {
      if (r.busy) continue;
      if (!got || r.holds(n)) got = &r;
      if (got->holds(n)) break;
    }
    if (!got) return nullptr;
    if (!got->holds(n)) {
      owed += gain;
      const double mb = HostStage::count(n) * HostStage::size(n) / 1048576.;
      if (owed < std::min(150. + 400. * mb, 1300.)) return nullptr;  // what pinning takes, us
    }
    got->busy = true;
    return got;
  }
  void give(HostStage* r) {
    std::lock_guard<std::mutex> lock(mu);
    r->busy = false;
  }
};
inline ReadPool& read_pool() {
  static ReadPool pool;
  return pool;
}
// A case or an ensemble, as long as it lives.
struct ReadPoolUser {
  ReadPool& pool;
  explicit ReadPoolUser(ReadPool& p = read_pool()) : pool(p) { pool.enter(); }
  ReadPoolUser(const ReadPoolUser&) = delete;
  ReadPoolUser& operator=(const ReadPoolUser&) = delete;
  ~ReadPoolUser() { pool.leave(); }
};
// what a read of n bytes gains by the pinned route, in us: one array, and values formed per cell
inline double array_gain(size_t n) { return n < HostStage::kArray ? 0. : 20. + n / 1048576. * 110.; }
inline double formed_gain(size_t n) { return 40. + n / 1048576. * 450.; }

// n bytes to dst through the ring's slots: fill(pinned, offset, length) enqueues one slot's worth on the
// stream.  Returns when dst is written.
template <class Fill>
hipError_t read_ring(HostStage& st, hipStream_t stream, char* dst, size_t n, Fill fill) {
  hipEvent_t ev[HostStage::kSlots] = {};
  hipError_t err = hipSuccess;
  for (int i = 0; i < st.slots && err == hipSuccess; ++i) err = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
  const int R = st.slots;
  const long nch = err == hipSuccess ? (long)((n + st.slot - 1) / st.slot) : 0;
  const int T = (int)std::min<size_t>(std::max<size_t>(n >> 21, 1), 8);  // pieces per chunk, and threads
  std::atomic<long> ready{0}, next{0};  // chunks in their slots; pieces taken
  std::atomic<bool> stop{false};
  std::atomic<int> left[HostStage::kSlots];
  auto copy = [&](long piece) {
    const long c = piece / T;
    const int t = (int)(piece % T);
    const size_t o = c * st.slot, len = std::min(st.slot, n - o);
    const size_t a = len * t / T & ~(size_t)63, b = t + 1 == T ? len : len * (t + 1) / T & ~(size_t)63;
    std::memcpy(dst + o + a, st.pin + (c % R) * st.slot + a, b - a);
    left[c % R].fetch_sub(1, std::memory_order_release);
  };
  auto help = [&] {
    for (;;) {
      const long p = next.fetch_add(1);
      if (p / T >= nch) return;
      while (ready.load(std::memory_order_acquire) <= p / T) {
        if (stop.load()) return;
        std::this_thread::yield();
      }
      copy(p);
    }
  };
  long issued = 0;
  auto issue = [&]() -> hipError_t {
    const size_t o = issued * st.slot;
    hipError_t e = fill(st.pin + (issued % R) * st.slot, o, std::min(st.slot, n - o));
    if (e == hipSuccess) e = hipEventRecord(ev[issued % R], stream);
    ++issued;
    return e;
  };
  while (err == hipSuccess && issued < nch && issued < R) err = issue();
  std::thread helpers[7];
  int nh = 0;
  if (err == hipSuccess) {
    try {
      for (; nh < T - 1; ++nh) helpers[nh] = std::thread(help);
    } catch (...) {  // no more threads: the ones there are do
    }
  }
  for (long c = 0; c < nch && err == hipSuccess; ++c) {
    err = hipEventSynchronize(ev[c % R]);
    if (err != hipSuccess) break;
    left[c % R].store(T);
    ready.store(c + 1, std::memory_order_release);
    for (long p = next.load(); p / T <= c;)
      if (next.compare_exchange_weak(p, p + 1)) {
        copy(p);
        p = next.load();
      }
    while (left[c % R].load(std::memory_order_acquire)) std::this_thread::yield();
    if (issued < nch) err = issue();
  }
  stop.store(true);
  for (int i = 0; i < nh; ++i) helpers[i].join();
  if (err != hipSuccess) (void)hipStreamSynchronize(stream);  // nothing still writes the slots
  for (hipEvent_t e : ev)
    if (e) (void)hipEventDestroy(e);
  return err;
}

// Makes a stream's device current for the calling thread (a new thread's is device 0): events are made
// and kernels launched there.
struct OnDeviceOf {
  int before = -1;
  explicit OnDeviceOf(hipStream_t s) {
    hipDevice_t d;
    int cur;
    if (hipStreamGetDevice(s, &d) == hipSuccess && hipGetDevice(&cur) == hipSuccess && d != cur &&
        hipSetDevice(d) == hipSuccess)
      before = cur;
  }
  OnDeviceOf(const OnDeviceOf&) = delete;
  OnDeviceOf& operator=(const OnDeviceOf&) = delete;
  ~OnDeviceOf() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

// n bytes to dst: by fill through a ring, or by plain().  `gain` as above; a gain of 0 is the plain route.
template <class Fill, class Plain>
hipError_t read_back(ReadPool& pool, hipStream_t stream, char* dst, size_t n, double gain, Fill fill, Plain plain) {
  if (!n) return hipSuccess;
  HostStage* r = gain > 0. ? pool.take(n, gain) : nullptr;
  if (!r) return plain();
  OnDeviceOf dev(stream);
  if (r->reserve(n) != hipSuccess) {  // pinned memory is not to be had
    pool.give(r);
    return plain();
  }
  const hipError_t e = read_ring(*r, stream, dst, n, fill);
  pool.give(r);
  return e;
}

// Cell c's value of a field that is formed per cell, as mahyco_get_field hands it out, from the cell's
// membership b and up to two arrays.  The membership itself; Materiau from the volume fraction g of a
// cell of one environment, else from those of its environments e [m][nc]; environment env's value: the
// cell value g in a cell of env alone, its own e (the volume: its fraction e of g) in a mixed cell, or
// g where it has none, 0 elsewhere.
MH_HD double field_value(int field, int env, int m, long nc, unsigned b, const double* g, const double* e, long c) {
  if (field == MH_F_ENV_MASK) return b;
  const bool pure = __builtin_popcount(b) == 1;
  if (field == MH_F_MATERIAU) {
    if (pure) return __builtin_ctz(b) * g[c];
    double val = 0.;
    for (int k = 0; k < m; ++k)
      if ((b >> k) & 1u) val += k * e[k * nc + c];
    return val;
  }
  if (env < 0 || !((b >> env) & 1u)) return 0.;
  if (pure || !e) return g[c];
  return field == MH_F_CELL_VOLUME ? e[c] * g[c] : e[c];
}
// n values from d, and those of cells c0 .. c0 + n - 1, to out.
template <int U = 0>
__global__ __launch_bounds__(MH_BLOCK) void k_read_array(const double* __restrict__ d, double* __restrict__ out, long n) {
  const long l = blockIdx.x * (long)MH_BLOCK + threadIdx.x;
  if (l < n) out[l] = d[l];
}
template <int U = 0>
__global__ __launch_bounds__(MH_BLOCK) void k_read_field(int field, int env, int m, long nc,
                                                         const uint8_t* __restrict__ mask, const double* __restrict__ g,
                                                         const double* __restrict__ e, double* __restrict__ out,
                                                         long c0, long n) {
  const long l = blockIdx.x * (long)MH_BLOCK + threadIdx.x;
  if (l < n) out[l] = field_value(field, env, m, nc, mask[c0 + l], g, e, c0 + l);
}

#endif
