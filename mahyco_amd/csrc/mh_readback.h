// mh_readback.h -- fields of the state to host memory.
//
// A copy to memory that is not pinned takes the runtime 165 us for 256 KB and 6.3 ms for 57 MB into
// pages not touched before (1.6 and 9 GB/s; the link does 56 GB/s into pinned memory).  Here the
// field goes through a ring of pinned slots, filled by the copy engine or, where the value is
// formed per cell, by a kernel that writes it there, and emptied by the calling thread and up to
// seven more: 68 us and 2.0 ms.  One thread below 4 MB (two copy 1 MB no faster than one), one more
// per 2 MB, eight at most (12 are slower); 4 MB slots at most (2 MB ones take 3.4 ms for 57 MB).
// The slots belong to a case or an ensemble, at most 16 MB, and are freed with it.  Threads that read
// fields of one case, or of the members of one ensemble, take turns.
#ifndef MH_READBACK_H
#define MH_READBACK_H

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "mh_state.h"

struct HostStage {
  static constexpr int kSlots = 4;
  std::mutex mu;  // held by a read from its first use of the slots to its last
  char* pin = nullptr;
  size_t slot = 0;  // bytes of a slot
  int slots = 0;
  hipEvent_t ev[kSlots] = {};

  hipError_t reserve(size_t n) {
    // small fields: one slot that holds them; larger ones: a quarter each, as far as 4 MB.  In powers
    // of two, so that a node field after a cell field of the same mesh, or one case of an ensemble
    // after another, seldom asks for more (pinning takes 0.1 to 0.6 ms)
    const int ns = n <= (256u << 10) ? 1 : kSlots;
    size_t want = 64u << 10;
    while (want * ns < n && want < (4u << 20)) want *= 2;
    if (pin && (size_t)slots * slot >= (size_t)ns * want) return hipSuccess;
    release();
    for (int i = 0; i < kSlots; ++i) {
      const hipError_t e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
      if (e != hipSuccess) {
        release();
        return e;
      }
    }
    hipError_t e = hipErrorOutOfMemory;
    for (size_t s = want; s >= 4096; s /= 2) {  // with less where pinned memory is short
      e = hipHostMalloc((void**)&pin, ns * s, hipHostMallocDefault);
      if (e == hipSuccess) {
        slot = s;
        slots = ns;
        return e;
      }
      pin = nullptr;
      (void)hipGetLastError();
    }
    release();
    return e;
  }
  void release() {
    if (pin) (void)hipHostFree(pin);
    for (auto& e : ev) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    pin = nullptr;
    slot = 0;
    slots = 0;
  }
  HostStage() = default;
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
  ~HostStage() { release(); }
};

// n bytes to dst: fill(pinned, offset, length) enqueues one slot's worth on the stream.  Returns
// when dst is written.
template <class Fill>
hipError_t read_back(HostStage& st, hipStream_t stream, char* dst, size_t n, Fill fill) {
  if (!n) return hipSuccess;
  std::lock_guard<std::mutex> turn(st.mu);
  hipError_t err = st.reserve(n);
  if (err != hipSuccess) return err;
  const int R = st.slots;
  const long nch = (long)((n + st.slot - 1) / st.slot);
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
    if (e == hipSuccess) e = hipEventRecord(st.ev[issued % R], stream);
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
    err = hipEventSynchronize(st.ev[c % R]);
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
  return err;
}

// Cell values as mahyco_get_field hands them out, cells c0 .. c0 + n - 1 to out.  Environment env's
// value is the cell value g in a cell of env alone, its own e (or g where there is none) in a mixed
// cell, 0 elsewhere; the volume and mass fractions, the volume and Materiau follow the same aliasing.
template <int U = 0>
__global__ __launch_bounds__(MH_BLOCK) void k_read_field(MhDev S, int field, int env, const double* __restrict__ g,
                                                         const double* __restrict__ e, double* __restrict__ out,
                                                         long c0, long n) {
  const long l = blockIdx.x * (long)MH_BLOCK + threadIdx.x;
  if (l >= n) return;
  const long c = c0 + l, nc = S.g.nc;
  const unsigned b = S.mask[c];
  const bool pure = __popc(b) == 1, in = env >= 0 && ((b >> env) & 1u);
  double val = 0.;
  if (field == MH_F_ENV_MASK) {
    val = b;
  } else if (field == MH_F_MATERIAU) {
    if (pure) {
      val = (__ffs(b) - 1) * S.fg[c];
    } else {
      for (int k = 0; k < S.m; ++k)
        if ((b >> k) & 1u) val += k * S.fk[k * nc + c];
    }
  } else if (field == MH_F_CELL_VOLUME) {
    if (env < 0) val = g[c];
    else if (in) val = pure ? g[c] : S.fk[env * nc + c] * g[c];
  } else if (field == MH_F_MASS_FRACTION) {
    if (in) val = pure ? S.chig[c] : S.chik[env * nc + c];
  } else {  // the volume fraction too: fg and fk
    if (env < 0) val = g[c];
    else if (in) val = pure || !e ? g[c] : e[c];
  }
  out[l] = val;
}

#endif
