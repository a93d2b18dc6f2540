// Caching allocator of page-locked host memory, for buffers that kernels and copy engines reach over PCIe directly: results
// that are read back (the last kernel of a read-back stores into the host tensor itself) and the staging block of a device.
// Page-locking costs hundreds of microseconds a call, so blocks are kept for reuse; both what is kept and what is handed out
// are bounded (alloc() returns null beyond that and the caller takes pageable memory), and release() gives back what is kept.
// What is kept follows the sizes in use: a block serves requests down to half its size, and the longest unused ones make room.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

namespace tt::runtime {

struct HostPoolBackend {
  int (*malloc)(void **ptr, size_t bytes);   // 0 on success
  int (*free)(void *ptr);
};

class HostPool {
public:
  static constexpr size_t kMaxCached = size_t(256) << 20;   // kept for reuse
  static constexpr size_t kMaxTotal = size_t(1) << 30;      // kept and in use together

  explicit HostPool(HostPoolBackend backend) : be(backend) {}

  // size classes an eighth of a power of two apart, so that results of slightly different sizes share blocks
  static size_t rounded(size_t bytes) {
    size_t step = 4096;
    while (step * 16 <= bytes) step *= 2;
    return std::max<size_t>(step, (bytes + step - 1) / step * step);
  }

  void *alloc(size_t bytes) {
    const size_t sz = rounded(bytes);
    std::vector<void *> gone;
    bool room;
    {
      std::lock_guard<std::mutex> g(mu);
      const auto it = kept.lower_bound({sz, 0});
      if (it != kept.end() && it->first.first <= 2 * sz) {
        void *p = it->second;
        inUse[p] = it->first.first;
        drop(it);
        return p;
      }
      while (total + sz > kMaxTotal && !kept.empty()) evict(gone);
      room = total + sz <= kMaxTotal;
      if (room) total += sz;
    }
    giveBack(gone);
    if (!room) return nullptr;
    void *p = nullptr;
    const bool got = be.malloc(&p, sz) == 0 && p;
    std::lock_guard<std::mutex> g(mu);
    if (got) inUse[p] = sz;
    else total -= sz;
    return got ? p : nullptr;
  }

  void free(void *p) {
    std::vector<void *> gone;
    {
      std::lock_guard<std::mutex> g(mu);
      const auto it = inUse.find(p);
      if (it == inUse.end()) return;
      const size_t sz = it->second;
      inUse.erase(it);
      if (sz > kMaxCached) {
        total -= sz;
        gone.push_back(p);
      } else {
        while (keptBytes + sz > kMaxCached) evict(gone);
        byAge[++clock] = sz;
        kept[{sz, clock}] = p;
        keptBytes += sz;
      }
    }
    giveBack(gone);
  }

  void release() {
    std::vector<void *> gone;
    {
      std::lock_guard<std::mutex> g(mu);
      while (!kept.empty()) evict(gone);
    }
    giveBack(gone);
  }

  size_t cached() {
    std::lock_guard<std::mutex> g(mu);
    return keptBytes;
  }

private:
  using Kept = std::map<std::pair<size_t, std::uint64_t>, void *>;   // (size, time it came back) -> block

  void drop(Kept::iterator it) {
    keptBytes -= it->first.first;
    byAge.erase(it->first.second);
    kept.erase(it);
  }
  void evict(std::vector<void *> &gone) {   // the block that has been kept for longest
    const auto oldest = byAge.begin();
    const auto it = kept.find({oldest->second, oldest->first});
    gone.push_back(it->second);
    total -= oldest->second;
    drop(it);
  }
  void giveBack(const std::vector<void *> &gone) {   // outside the lock: an unlock takes as long as a page-lock
    for (void *p : gone) be.free(p);
  }

  HostPoolBackend be;
  std::mutex mu;
  Kept kept;
  std::map<std::uint64_t, size_t> byAge;
  std::unordered_map<void *, size_t> inUse;
  std::uint64_t clock = 0;
  size_t keptBytes = 0, total = 0;
};

}  // namespace tt::runtime
