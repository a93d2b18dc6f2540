// Copies between host buffers of several MiB, shared with a few helper threads: one core moves what a device has just written
// into fresh pages at 30 GB/s, which is less than PCIe delivers ([2048, 4096] bf16, 16 MiB: 0.55 ms of the 1.4 ms a read-back
// took), mostly in page faults and cache misses that further cores take beside it.
#pragma once
#include <unistd.h>

#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>

namespace tt::runtime {

class HostCopy {
public:
  static constexpr size_t kChunk = size_t(256) << 10;
  static constexpr size_t kShareFrom = size_t(1) << 20;   // below, waking a helper takes as long as the copy
  static constexpr int kHelpers = 5;

  // Returns when all bytes are there.  The caller takes chunks as the helpers do, so it never waits for a thread that has not
  // been scheduled: only for chunks that were begun.  A forked child has neither the helpers nor a lock and a condition variable it
  // could rely on, and copies alone.
  static void run(void *dst, const void *src, size_t bytes) {
    if (bytes < kShareFrom) {
      std::memcpy(dst, src, bytes);
      return;
    }
    static HostCopy *crew = new HostCopy;   // never destroyed: its threads wait until the process ends
    if (crew->owner != getpid()) std::memcpy(dst, src, bytes);
    else crew->share(dst, src, bytes);
  }

private:
  struct Job {
    std::uint8_t *dst;
    const std::uint8_t *src;
    size_t bytes, chunks;
    std::atomic<size_t> next{0}, done{0};
    void work() {
      for (size_t i; (i = next.fetch_add(1, std::memory_order_relaxed)) < chunks;) {
        const size_t at = i * kChunk, n = bytes - at < kChunk ? bytes - at : kChunk;
        std::memcpy(dst + at, src + at, n);
        done.fetch_add(1, std::memory_order_release);
      }
    }
  };

  HostCopy() {
    const unsigned cores = std::thread::hardware_concurrency();
    const int n = cores < 2 ? 0 : static_cast<int>(cores / 2 < kHelpers ? cores / 2 : kHelpers);
    try {
      for (int i = 0; i < n; ++i) std::thread([this] { serve(); }).detach();
    } catch (const std::system_error &) {   // no more threads to be had: the caller copies with those there are, or alone
    }
  }
  void serve() {
    std::uint64_t seen = 0;
    for (;;) {
      std::shared_ptr<Job> j;
      {
        std::unique_lock<std::mutex> g(mu);
        cv.wait(g, [&] { return turn != seen; });
        seen = turn;
        j = job;
      }
      if (j) j->work();
    }
  }
  void share(void *dst, const void *src, size_t bytes) {
    auto j = std::make_shared<Job>();
    j->dst = static_cast<std::uint8_t *>(dst);
    j->src = static_cast<const std::uint8_t *>(src);
    j->bytes = bytes;
    j->chunks = (bytes + kChunk - 1) / kChunk;
    {
      std::lock_guard<std::mutex> g(mu);   // a copy of another thread in progress keeps the helpers it has
      job = j;
      ++turn;
    }
    cv.notify_all();
    j->work();
    while (j->done.load(std::memory_order_acquire) != j->chunks) std::this_thread::yield();
    std::lock_guard<std::mutex> g(mu);
    if (job == j) job.reset();
  }

  const pid_t owner = getpid();
  std::mutex mu;
  std::condition_variable cv;
  std::shared_ptr<Job> job;
  std::uint64_t turn = 0;
};

}  // namespace tt::runtime
