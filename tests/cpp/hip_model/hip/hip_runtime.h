// A model of the few HIP runtime calls that public_amd/csrc/host_copy.hpp makes,
// for CPU checks of its bookkeeping: several devices, streams and events that
// belong to one each (an event is recorded on streams of its own device only),
// and counts of what is alive.  Memory of every device is host memory.
#pragma once
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <thread>

#define __global__
#define __launch_bounds__(n)
struct ModelDim {
  unsigned x = 0, y = 0, z = 0;
};
static ModelDim blockIdx, blockDim, gridDim, threadIdx;

typedef int hipError_t;
constexpr hipError_t hipSuccess = 0, hipErrorInvalidHandle = 400;
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
constexpr unsigned hipHostMallocPortable = 1, hipEventDisableTiming = 2;
struct ModelStream {
  int device;
};
struct ModelEvent {
  int device;
};
typedef ModelStream *hipStream_t;
typedef ModelEvent *hipEvent_t;

static thread_local int model_device = 0;
static std::atomic<int> model_events{0}, model_pinned{0}, model_recorded{0}, model_no_events{0};
static std::atomic<bool> model_hold{false}, model_held{false};

inline hipError_t hipSetDevice(int d) {
  model_device = d;
  return hipSuccess;
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::malloc(n);
  ++model_pinned;
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  std::free(p);
  --model_pinned;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  if (model_no_events) return 2;  // out of memory
  *e = new ModelEvent{model_device};
  ++model_events;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  delete e;
  --model_events;
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  if (e->device != s->device) return hipErrorInvalidHandle;
  ++model_recorded;
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  while (model_hold) {  // a transfer that takes its time
    model_held = true;
    std::this_thread::sleep_for(std::chrono::milliseconds(1));
  }
  std::memcpy(d, s, n);
  return hipSuccess;
}
