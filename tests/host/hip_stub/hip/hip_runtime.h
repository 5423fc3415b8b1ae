// Stand-in for the HIP calls of mh_readback.h, so that its host side runs on a CPU: streams run
// everything at once, pinned memory is ordinary memory and is overwritten before it is freed.
#ifndef MH_HIP_STUB_H
#define MH_HIP_STUB_H
#include <atomic>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#define __global__
#define __device__
#define __host__
#define __launch_bounds__(...)

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorInvalidHandle = 400 };
struct StubStream {
  int device = 0;
};
struct StubEvent {
  int device = 0;
};
typedef StubStream* hipStream_t;
typedef StubEvent* hipEvent_t;
typedef int hipDevice_t;
enum { hipEventDisableTiming = 2, hipHostMallocDefault = 0, hipHostMallocPortable = 1 };

// Each thread has a current device, 0 at first; an event belongs to the device that was current when it
// was made, and only a stream of that device can record it.
static thread_local int stub_device = 0;
static inline hipError_t hipGetDevice(int* d) {
  *d = stub_device;
  return hipSuccess;
}
static inline hipError_t hipSetDevice(int d) {
  stub_device = d;
  return hipSuccess;
}
static inline hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
  *d = s ? s->device : stub_device;
  return hipSuccess;
}

struct StubDim {
  unsigned x = 0, y = 0, z = 0;
};
static thread_local StubDim blockIdx, threadIdx;

static size_t stub_head = 64;  // the size of an allocation lies ahead of it
static std::atomic<long> stub_pins{0}, stub_pinned{0};  // allocations made, bytes held
static size_t stub_most = ~(size_t)0;  // bytes that can be pinned at once
static inline hipError_t hipHostMalloc(void** p, size_t n, unsigned = 0) {
  char* b = n <= stub_most ? (char*)std::malloc(n + stub_head) : nullptr;
  if (!b) return hipErrorOutOfMemory;
  std::memcpy(b, &n, sizeof n);
  *p = b + stub_head;
  ++stub_pins;
  stub_pinned += (long)n;
  return hipSuccess;
}
static inline hipError_t hipHostFree(void* p) {
  char* b = (char*)p - stub_head;
  size_t n;
  std::memcpy(&n, b, sizeof n);
  std::memset(p, 0xee, n);
  stub_pinned -= (long)n;
  std::free(b);
  return hipSuccess;
}
static inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = new StubEvent{stub_device};
  return hipSuccess;
}
static inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  return hipSuccess;
}
static inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  return e->device == s->device ? hipSuccess : hipErrorInvalidHandle;
}
static inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
static inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
static inline hipError_t hipGetLastError() { return hipSuccess; }
#endif
