// The staged host copies of public_amd/csrc/host_copy.hpp over the HIP model of
// hip_model/: contexts of several devices, users that come and go meanwhile.
// Prints one line per case: name ok.
#include <algorithm>
#include <cstdio>
#include <future>
#include <vector>

#include "../../public_amd/csrc/host_copy.hpp"

using namespace cruna;

static bool round_trip(int device, size_t bytes, unsigned seed) {
  ModelStream s{device};
  std::vector<char> a(bytes), dev(bytes, 0), b(bytes, 0);
  for (size_t i = 0; i < bytes; ++i) a[i] = (char)((i * 2654435761u + seed) >> 13);
  HostCopyPool &pool = HostCopyPool::get();
  return pool.copy(dev.data(), a.data(), bytes, true, device, &s) == hipSuccess &&
         pool.copy(b.data(), dev.data(), bytes, false, device, &s) == hipSuccess && a == b;
}

int main() {
  const size_t sizes[] = {HC_MIN_TO_HOST + 8, HC_MIN_TO_DEVICE + 24};
  bool ok = true;
  {
    HostCopyUser u;
    // a context of each device, in turn
    for (int device : {0, 1, 0, 2, 1})
      for (size_t n : sizes) ok = ok && round_trip(device, n, device + 1);
    std::printf("devices %d\n", ok && model_recorded > 0);
    std::printf("events_bounded %d\n", model_events <= HC_THREADS);
    // no event can be made: the copy takes the plain path
    model_no_events = 1;
    std::printf("no_events %d\n", round_trip(5, sizes[1], 9));
    model_no_events = 0;
    std::printf("events_again %d\n", round_trip(5, sizes[1], 9));
    // while one copy runs, contexts come and go without waiting for it
    std::vector<char> a(sizes[1], 1), dev(sizes[1]);
    ModelStream s{0};
    model_held = false;
    model_hold = true;
    auto copy = std::async(std::launch::async, [&] {
      return HostCopyPool::get().copy(dev.data(), a.data(), a.size(), true, 0, &s);
    });
    while (!model_held) std::this_thread::yield();
    auto other = std::async(std::launch::async, [] { HostCopyUser v; });
    const bool free = other.wait_for(std::chrono::seconds(5)) == std::future_status::ready;
    model_hold = false;
    other.wait();
    std::printf("users_do_not_wait %d\n", free && copy.get() == hipSuccess && a == dev);
  }
  std::printf("given_back %d\n", model_events == 0 && model_pinned == 0);
  {
    HostCopyUser u;
    std::printf("made_again %d\n", round_trip(1, sizes[1], 3) && model_pinned > 0);
  }
  std::printf("given_back_again %d\n", model_events == 0 && model_pinned == 0);
  return 0;
}
