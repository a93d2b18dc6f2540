// Caching allocator of page-locked host memory, for buffers that kernels and copy engines reach over PCIe directly: results
// that are read back (the last kernel of a read-back stores into the host tensor itself) and the staging block of a device.
// Page-locking costs hundreds of microseconds a call, so blocks are kept for reuse; both what is kept and what is handed out
// are bounded (alloc() returns null beyond that and the caller takes pageable memory), and release() gives back what is kept.
#pragma once
#include <algorithm>
#include <cstddef>
#include <map>
#include <mutex>

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
    {
      std::lock_guard<std::mutex> g(mu);
      auto it = kept.find(sz);
      if (it != kept.end()) {
        void *p = it->second;
        kept.erase(it);
        keptBytes -= sz;
        return p;
      }
      if (total + sz > kMaxTotal) return nullptr;
      total += sz;
    }
    void *p = nullptr;
    if (be.malloc(&p, sz) == 0 && p) return p;
    std::lock_guard<std::mutex> g(mu);
    total -= sz;
    return nullptr;
  }

  void free(void *p, size_t bytes) {
    const size_t sz = rounded(bytes);
    {
      std::lock_guard<std::mutex> g(mu);
      if (keptBytes + sz <= kMaxCached) {
        kept.emplace(sz, p);
        keptBytes += sz;
        return;
      }
      total -= sz;
    }
    be.free(p);
  }

  void release() {
    std::multimap<size_t, void *> gone;
    {
      std::lock_guard<std::mutex> g(mu);
      gone.swap(kept);
      total -= keptBytes;
      keptBytes = 0;
    }
    for (auto &kv : gone) be.free(kv.second);
  }

private:
  HostPoolBackend be;
  std::mutex mu;
  std::multimap<size_t, void *> kept;
  size_t keptBytes = 0, total = 0;
};

}  // namespace tt::runtime
