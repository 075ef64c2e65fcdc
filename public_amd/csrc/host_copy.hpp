// Copies between pageable host arrays and the device, and the padded layout.
//
// A copy to or from pageable memory goes through the runtime's own staging
// buffer with one CPU thread (10 GB/s measured for a 671 MB state, most of it
// the thread's memcpy and the first touch of the destination's pages), which
// was 18 % of 25 steps at 256^3 and a third of an optimisation iteration at 128^3.
// Large copies here run through pinned chunks with several threads: a thread
// moves its chunks between the host array and its pinned chunk while other
// threads' chunks are on the bus.  The pinned memory (32 MB) belongs to
// a process-wide pool that is made with the first large copy, used by one copy at
// a time (a copy that finds it busy takes the plain path) and freed with the
// last context or closure.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace cruna {

constexpr int HC_THREADS = 8;
constexpr size_t HC_CHUNK = 4u << 20;  // bytes of a pinned chunk
// Smallest staged copies.  To the host the plain path also touches the new
// array's pages, and starting the threads pays from 8 MB on (an RHS call on 11 MB
// arrays 1.24 -> 0.99 ms); to the device it does not for arrays of 10 MB (two of
// them 0.06 ms slower).
constexpr size_t HC_MIN_TO_HOST = 8u << 20, HC_MIN_TO_DEVICE = 32u << 20;

class HostCopyPool {
 public:
  static HostCopyPool &get() {
    static HostCopyPool *p = new HostCopyPool();  // outlives every user
    return *p;
  }
  // (a count of its own: no context waits for another one's copy when it is
  // made or released)
  void add_user() { ++users_; }
  void drop_user() {
    if (--users_ > 0) return;
    // nobody copies any more, unless a user came since: its own end gives back then
    std::lock_guard<std::mutex> l(mu_);
    if (users_ == 0) give_back();
  }
  // host <-> dev on stream s of device `device`.  The host array may be used
  // again (to the device) or holds the values (to the host) when it returns.
  hipError_t copy(void *dst, const void *src, size_t bytes, bool to_device, int device, hipStream_t s) {
    const hipMemcpyKind kind = to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
    if (bytes >= (to_device ? HC_MIN_TO_DEVICE : HC_MIN_TO_HOST)) {
      std::unique_lock<std::mutex> l(mu_, std::try_to_lock);
      if (l.owns_lock() && reserve()) {
        hipError_t e = hipSuccess;
        if (staged(dst, src, bytes, to_device, device, s, e)) return e;
      }
    }
    hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
    // (the runtime has staged a pageable source when its copy call returns)
    if (e == hipSuccess && !to_device) e = hipStreamSynchronize(s);
    return e;
  }

 private:
  // A thread's chunk, which any device reaches, and the event of its last
  // transfer: an event belongs to one device and is recorded on that device's
  // streams only, so it is made anew when the slot serves another one.
  struct Slot {
    void *pin = nullptr;
    hipEvent_t ev = nullptr;
    int device = -1;  // of ev
    hipError_t bind(int d) {
      hipError_t e = hipSetDevice(d);
      if (e != hipSuccess || (ev && device == d)) return e;
      if (ev) (void)hipEventDestroy(ev);
      ev = nullptr;
      e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
      if (e != hipSuccess) ev = nullptr;
      device = d;
      return e;
    }
  };
  std::mutex mu_;  // held by the copy that uses the slots
  std::atomic<int> users_{0};
  Slot slots_[HC_THREADS];

  void give_back() {
    for (auto &s : slots_) {
      if (s.ev) (void)hipEventDestroy(s.ev);
      if (s.pin) (void)hipHostFree(s.pin);
      s = Slot{};
    }
  }
  bool reserve() {
    if (slots_[HC_THREADS - 1].pin) return true;
    for (auto &s : slots_)
      if (hipHostMalloc(&s.pin, HC_CHUNK, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        s.pin = nullptr;
        give_back();
        return false;
      }
    return true;
  }

  // false: no thread could be started or made its event, nothing was copied
  bool staged(void *dst, const void *src, size_t bytes, bool to_device, int device, hipStream_t s, hipError_t &err) {
    const int nt = (int)std::min<size_t>(HC_THREADS, std::max<size_t>(2, bytes / HC_CHUNK));
    // at least two chunks per thread, so that copies and transfers overlap
    size_t chunk = (bytes / (2 * nt) + 4095) / 4096 * 4096;
    chunk = std::min(HC_CHUNK, std::max<size_t>(chunk, 4096));
    const size_t n = (bytes + chunk - 1) / chunk;
    std::atomic<size_t> next{0};
    std::atomic<int> bad{(int)hipSuccess}, ready{0};
    auto work = [&](int t) {
      Slot &slot = slots_[t];
      hipError_t e = slot.bind(device);
      if (e != hipSuccess) return;  // the other threads share out its chunks
      ++ready;
      bool used = false;
      while (e == hipSuccess && bad.load() == (int)hipSuccess) {
        const size_t i = next.fetch_add(1);
        if (i >= n) break;
        const size_t at = i * chunk, len = std::min(chunk, bytes - at);
        if (to_device) {
          if (used) e = hipEventSynchronize(slot.ev);  // the chunk's last transfer
          if (e != hipSuccess) break;
          std::memcpy(slot.pin, (const char *)src + at, len);
          e = hipMemcpyAsync((char *)dst + at, slot.pin, len, hipMemcpyHostToDevice, s);
          if (e == hipSuccess) e = hipEventRecord(slot.ev, s);
          used = true;
        } else {
          e = hipMemcpyAsync(slot.pin, (const char *)src + at, len, hipMemcpyDeviceToHost, s);
          if (e == hipSuccess) e = hipEventRecord(slot.ev, s);
          if (e == hipSuccess) e = hipEventSynchronize(slot.ev);
          if (e == hipSuccess) std::memcpy((char *)dst + at, slot.pin, len);
        }
      }
      if (used && e == hipSuccess) e = hipEventSynchronize(slot.ev);
      if (e != hipSuccess) {
        int none = (int)hipSuccess;
        bad.compare_exchange_strong(none, (int)e);
      }
    };
    std::vector<std::thread> th;
    try {
      th.reserve(nt);
      for (int t = 0; t < nt; ++t) th.emplace_back(work, t);
    } catch (const std::exception &) {
      // the threads that did start share out all chunks
      if (th.empty()) return false;
    }
    for (auto &t : th) t.join();
    if (ready.load() == 0) return false;
    err = (hipError_t)bad.load();
    if (err != hipSuccess) (void)hipStreamSynchronize(s);  // nothing uses the pinned chunks any more
    return true;
  }
};

// Keeps the pool alive (a member of what copies through it).
struct HostCopyUser {
  HostCopyUser() { HostCopyPool::get().add_user(); }
  ~HostCopyUser() { HostCopyPool::get().drop_user(); }
  HostCopyUser(const HostCopyUser &) = delete;
  HostCopyUser &operator=(const HostCopyUser &) = delete;
};

// Fields in the padded device layout (p1, p2, p3) with (f1, f2, f3) points in
// front of the n1 x n2 x n3 real ones.
struct PadLayout {
  int n1, n2, n3, p1, p2, p3, f1, f2, f3;
};
struct PadFill {
  double v[5];
};

// Real points (contiguous, Fortran order) of nv fields into the padded layout,
// padding points set to fill.v[field].
__global__ __launch_bounds__(256) void k_scatter_real(const double *__restrict__ src, double *__restrict__ dst, int nv,
                                                      PadLayout l, PadFill fill) {
  const long N = (long)l.p1 * l.p2 * l.p3, Nr = (long)l.n1 * l.n2 * l.n3;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < nv * N; t += (long)gridDim.x * blockDim.x) {
    const int v = (int)(t / N);
    const long p = t - v * N;
    const int i = (int)(p % l.p1) - l.f1, j = (int)((p / l.p1) % l.p2) - l.f2, k = (int)(p / ((long)l.p1 * l.p2)) - l.f3;
    const bool real = i >= 0 && i < l.n1 && j >= 0 && j < l.n2 && k >= 0 && k < l.n3;
    dst[t] = real ? src[v * Nr + i + (long)l.n1 * (j + (long)l.n2 * k)] : fill.v[v];
  }
}

// The real points of nv padded fields (type T) into a contiguous FP64 array.
template <typename T>
__global__ __launch_bounds__(256) void k_gather_real(const T *__restrict__ src, double *__restrict__ dst, int nv,
                                                     PadLayout l) {
  const long N = (long)l.p1 * l.p2 * l.p3, Nr = (long)l.n1 * l.n2 * l.n3;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < nv * Nr; t += (long)gridDim.x * blockDim.x) {
    const int v = (int)(t / Nr);
    const long r = t - v * Nr;
    const int i = (int)(r % l.n1), j = (int)((r / l.n1) % l.n2), k = (int)(r / ((long)l.n1 * l.n2));
    dst[t] = double(src[v * N + (i + l.f1) + (long)l.p1 * ((j + l.f2) + (long)l.p2 * (k + l.f3))]);
  }
}

}  // namespace cruna
