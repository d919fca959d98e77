#include "devmem.hpp"
#include <algorithm>
#include <cstdint>
#include <map>
#include <mutex>
#include <new>
#include <vector>

namespace tvk {
namespace {

struct Block {
  void* p;
  size_t bytes;
};
struct Kept {
  std::vector<Block> blocks;   // the longest kept first
  size_t bytes = 0, limit = 0;
  int users = 0;
  uint64_t trims = 0;          // how often the blocks were freed
};
constexpr size_t kMaxBlocks = 16;

std::mutex g_mu;
std::map<int, Kept>& kept() {
  // never destroyed: blocks may go back while the process ends
  static std::map<int, Kept>* m = new std::map<int, Kept>;
  return *m;
}

// frees every kept block of the device (g_mu held); false when there was none
bool trim(Kept& k) {
  if (k.blocks.empty()) return false;
  for (const Block& b : k.blocks) (void)hipFree(b.p);
  k.blocks.clear();
  k.bytes = 0;
  ++k.trims;
  return true;
}

void give_back(int device, void* p, size_t bytes, bool idle) {
  int cur = device;
  (void)hipGetDevice(&cur);
  if (cur != device) (void)hipSetDevice(device);
  bool keep = false;
  if (idle || hipDeviceSynchronize() == hipSuccess) {
    std::lock_guard<std::mutex> lk(g_mu);
    Kept& k = kept()[device];
    if (k.users > 0 && bytes <= k.limit) {
      while (!k.blocks.empty() && (k.blocks.size() >= kMaxBlocks || k.bytes + bytes > k.limit)) {
        (void)hipFree(k.blocks.front().p);
        k.bytes -= k.blocks.front().bytes;
        k.blocks.erase(k.blocks.begin());
      }
      try {
        k.blocks.push_back(Block{p, bytes});
        k.bytes += bytes;
        keep = true;
      } catch (const std::bad_alloc&) {
      }
    }
  }
  if (!keep) (void)hipFree(p);
  if (cur != device) (void)hipSetDevice(cur);
}

struct GiveBack {
  int device;
  size_t bytes;
  bool idle = false;
  void operator()(void* p) const { give_back(device, p, bytes, idle); }
};

}  // namespace

hipError_t device_alloc_bytes(void** p, size_t bytes) {
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  uint64_t seen;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    seen = kept()[device].trims;
  }
  for (;;) {
    e = hipMalloc(p, bytes);
    if (e != hipErrorOutOfMemory) return e;
    {
      std::lock_guard<std::mutex> lk(g_mu);
      Kept& k = kept()[device];
      // nothing to free now, nor freed by another thread since this one last tried
      if (!trim(k) && k.trims == seen) return e;
      seen = k.trims;
    }
    (void)hipGetLastError();
  }
}

hipError_t device_block(std::shared_ptr<void>* out, size_t bytes, std::shared_ptr<void>* spare) {
  out->reset();
  int device = 0;
  hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  // whole 64 KiB, so that small tables of about one size share a block
  size_t want = (std::max<size_t>(bytes, 1) + 0xffff) & ~(size_t)0xffff;
  void* p = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    Kept& k = kept()[device];
    size_t best = k.blocks.size();
    for (size_t i = 0; i < k.blocks.size(); ++i)
      if (k.blocks[i].bytes >= want && k.blocks[i].bytes - want <= want / 8 &&
          (best == k.blocks.size() || k.blocks[i].bytes < k.blocks[best].bytes))
        best = i;
    if (best < k.blocks.size()) {
      p = k.blocks[best].p;
      want = k.blocks[best].bytes;
      k.bytes -= want;
      k.blocks.erase(k.blocks.begin() + (std::ptrdiff_t)best);
    }
  }
  if (!p) {
    e = device_alloc_bytes(&p, want);
    if (e == hipErrorOutOfMemory && spare && *spare) {
      (void)hipGetLastError();
      spare->reset();   // kept, and freed by the next attempt
      e = device_alloc_bytes(&p, want);
    }
    if (e != hipSuccess) return e;
  }
  *out = std::shared_ptr<void>(p, GiveBack{device, want});
  return hipSuccess;
}

void device_idle(const std::shared_ptr<void>& block) {
  if (GiveBack* g = std::get_deleter<GiveBack>(block)) g->idle = true;
}

void device_hold(int device) {
  std::lock_guard<std::mutex> lk(g_mu);
  Kept& k = kept()[device];
  ++k.users;
  if (k.limit == 0) {
    size_t total = 0;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) == hipSuccess) total = prop.totalGlobalMem;
    k.limit = total / 16;
  }
}

void device_release(int device) {
  std::lock_guard<std::mutex> lk(g_mu);
  (void)trim(kept()[device]);
}

void device_drop(int device) {
  std::lock_guard<std::mutex> lk(g_mu);
  Kept& k = kept()[device];
  if (--k.users <= 0) {
    k.users = 0;
    (void)trim(k);
  }
}

}  // namespace tvk
