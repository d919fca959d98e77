// Checks of the dataset memory (tuvok_amd/csrc/devmem.cpp) over a pretended device
// of 1 MiB x 1024: what happens when it is full.  Prints "ok".
#include <hip/hip_runtime.h>
#include <atomic>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <mutex>
#include <thread>
#include <vector>
#include "devmem.hpp"

static std::mutex g;
static std::condition_variable cv;
static std::map<void*, size_t> live;
static size_t used = 0;
static const size_t kTotal = size_t(1) << 30, MB = size_t(1) << 20;
static std::atomic<int> hold_failures{0};   // so many failed calls wait for each other before they return
static int waiting = 0;

hipError_t hipMalloc(void** p, size_t bytes) {
  std::unique_lock<std::mutex> lk(g);
  if (used + bytes > kTotal) {
    if (hold_failures > 0) {
      const int want = hold_failures;
      if (++waiting >= want) { hold_failures = 0; cv.notify_all(); }
      cv.wait(lk, [] { return hold_failures == 0; });
    }
    return hipErrorOutOfMemory;
  }
  *p = std::malloc(1);
  live[*p] = bytes;
  used += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  std::lock_guard<std::mutex> lk(g);
  auto it = live.find(p);
  if (it == live.end()) return hipErrorInvalidValue;
  used -= it->second;
  live.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) { p->totalGlobalMem = kTotal; return hipSuccess; }

#define CHECK(x)                                                          \
  do {                                                                    \
    if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; }   \
  } while (0)

using namespace tvk;

// Two threads find the device full, both before either gives back what is kept:
// both get their memory from it.
static int two_threads_out_of_memory() {
  device_hold(0);
  {
    std::shared_ptr<void> a;
    CHECK(device_block(&a, 60 * MB) == hipSuccess);
    a.reset();   // kept: 60 of at most 64 MiB
    void* rest = nullptr;
    CHECK(hipMalloc(&rest, 944 * MB) == hipSuccess);   // 20 MiB are free
    hold_failures = 2;
    waiting = 0;
    hipError_t e[2];
    void* p[2] = {nullptr, nullptr};
    std::vector<std::thread> ts;
    for (int i = 0; i < 2; ++i) ts.emplace_back([&, i] { e[i] = device_alloc_bytes(&p[i], 30 * MB); });
    for (auto& t : ts) t.join();
    CHECK(e[0] == hipSuccess && e[1] == hipSuccess);
    void* more = nullptr;
    CHECK(device_alloc_bytes(&more, 30 * MB) == hipErrorOutOfMemory);   // and nothing is left to give back
    for (void* q : {p[0], p[1], rest}) CHECK(hipFree(q) == hipSuccess);
  }
  device_drop(0);
  CHECK(used == 0);
  return 0;
}

// A block that does not fit takes the room of one the caller can do without, and
// leaves it alone where there is room.
static int spare_block() {
  device_hold(0);
  {
    void* rest = nullptr;
    std::shared_ptr<void> spare, a, b;
    CHECK(device_block(&spare, 70 * MB) == hipSuccess);   // larger than what may be kept
    CHECK(hipMalloc(&rest, 904 * MB) == hipSuccess);   // 50 MiB are free
    CHECK(device_block(&a, 10 * MB, &spare) == hipSuccess && spare);
    CHECK(device_block(&b, 100 * MB, &spare) == hipSuccess && !spare);
    std::shared_ptr<void> c;
    CHECK(device_block(&c, 100 * MB, &spare) == hipErrorOutOfMemory && !c);
    CHECK(device_block(&spare, 5 * MB) == hipSuccess);
    CHECK(device_block(&c, 8 * MB, &spare) == hipSuccess && !spare);   // 10 MiB with the spare's, which was kept
    CHECK(hipFree(rest) == hipSuccess);
  }
  device_drop(0);
  CHECK(used == 0);
  return 0;
}

// What is kept goes when asked for; blocks in use stay.
static int release() {
  device_hold(0);
  {
    std::shared_ptr<void> a, b;
    CHECK(device_block(&a, 20 * MB) == hipSuccess && device_block(&b, 30 * MB) == hipSuccess);
    device_idle(a);
    a.reset();
    CHECK(used == 50 * MB);
    device_release(0);
    CHECK(used == 30 * MB);
  }
  CHECK(used == 30 * MB);
  device_drop(0);
  CHECK(used == 0);
  return 0;
}

int main() {
  if (release()) return 1;
  if (spare_block()) return 1;
  if (two_threads_out_of_memory()) return 1;
  std::printf("ok\n");
  return 0;
}
