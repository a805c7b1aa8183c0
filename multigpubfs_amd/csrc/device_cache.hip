// Device memory kept between batch engines.  A sweep creates an engine,
// admits hundreds of instances and drops it; handing its arena back to the
// driver costs nothing at first, but memory freed before has to be cleared
// before it is handed out again: in a process that had used 100 GB a sweep of
// 42 ms took 450 ms, almost all of it inside hipMalloc.  Whole arena chunks
// are kept instead, at most kKept bytes per device, and given back when an
// allocation of this library fails or mgbfs_release_cached_memory is called;
// budgets taken from free memory count them as free.
//
// A chunk is put here only after its engine's streams are idle, and taken by
// one engine at a time, so no order between streams is needed.
#include <mutex>
#include <vector>
#include "engine.hpp"

namespace mgbfs {

namespace {

constexpr uint64_t kKept = 16ull << 30;

struct Kept {
  int device;
  DeviceBuffer buf;
};

struct Cache {
  std::mutex mutex;
  std::vector<Kept> kept;
};

// Never destroyed: the runtime may be gone when static objects are.
Cache& cache() {
  static Cache* c = new Cache;
  return *c;
}

}  // namespace

DeviceBuffer device_cache_take(int device, uint64_t least, uint64_t most) {
  Cache& c = cache();
  std::lock_guard<std::mutex> lock(c.mutex);
  size_t best = c.kept.size();
  for (size_t k = 0; k < c.kept.size(); ++k)
    if (c.kept[k].device == device && c.kept[k].buf.bytes() >= least && c.kept[k].buf.bytes() <= most &&
        (best == c.kept.size() || c.kept[k].buf.bytes() < c.kept[best].buf.bytes()))
      best = k;
  DeviceBuffer out;
  if (best < c.kept.size()) {
    out = std::move(c.kept[best].buf);
    c.kept.erase(c.kept.begin() + static_cast<std::ptrdiff_t>(best));
  }
  return out;
}

void device_cache_give(int device, DeviceBuffer&& buf) {
  DeviceBuffer mine = std::move(buf);  // freed here when it is not kept
  Cache& c = cache();
  std::lock_guard<std::mutex> lock(c.mutex);
  uint64_t held = mine.bytes();
  for (const Kept& k : c.kept)
    if (k.device == device) held += k.buf.bytes();
  if (held <= kKept) c.kept.push_back(Kept{device, std::move(mine)});
}

uint64_t device_cache_bytes(int device) {
  Cache& c = cache();
  std::lock_guard<std::mutex> lock(c.mutex);
  uint64_t held = 0;
  for (const Kept& k : c.kept)
    if (k.device == device) held += k.buf.bytes();
  return held;
}

bool device_cache_release(int device) {
  std::vector<Kept> out;
  Cache& c = cache();
  std::lock_guard<std::mutex> lock(c.mutex);
  for (size_t k = c.kept.size(); k-- > 0;)
    if (c.kept[k].device == device) {
      out.push_back(std::move(c.kept[k]));
      c.kept.erase(c.kept.begin() + static_cast<std::ptrdiff_t>(k));
    }
  return !out.empty();
}

}  // namespace mgbfs

extern "C" void mgbfs_release_cached_memory(int32_t device) { (void)mgbfs::device_cache_release(device); }
