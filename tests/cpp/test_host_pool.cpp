// Host-side checks of the page-locked pool's bookkeeping with malloc / free standing in for the driver.
// Build: g++ -std=c++17 -I tt-mlir_amd/runtime tests/cpp/test_host_pool.cpp -o <exe>; exit status 0 = all checks passed.
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

#include "host_pool.h"

using tt::runtime::HostPool;
using tt::runtime::HostPoolBackend;

static std::set<void *> g_driver;   // blocks the "driver" has handed out and not taken back
static int g_locks = 0, g_unlocks = 0, g_fail_next = 0;

static int mockMalloc(void **p, size_t) {   // the pool never touches the memory: addresses are enough
  if (g_fail_next > 0) { --g_fail_next; *p = nullptr; return 1; }
  *p = std::malloc(1);
  g_driver.insert(*p);
  ++g_locks;
  return 0;
}
static int mockFree(void *p) {
  if (!g_driver.erase(p)) { std::fprintf(stderr, "double free or foreign pointer %p\n", p); std::abort(); }
  std::free(p);
  ++g_unlocks;
  return 0;
}

#define CHECK(cond)                                                          \
  do {                                                                       \
    if (!(cond)) { std::fprintf(stderr, "%s:%d: CHECK(%s) failed\n", __FILE__, __LINE__, #cond); return 1; } \
  } while (0)

static const size_t MiB = size_t(1) << 20;

static int reuse() {
  HostPool pool(HostPoolBackend{mockMalloc, mockFree});
  void *a = pool.alloc(1000000);
  pool.free(a);
  void *b = pool.alloc(1040000);            // the same size class
  CHECK(b == a);
  pool.free(b);
  void *c = pool.alloc(600000);             // more than half of the kept block
  CHECK(c == a && pool.cached() == 0);
  pool.free(c);
  CHECK(pool.cached() == HostPool::rounded(1000000));   // counted with its own size
  void *d = pool.alloc(100000);             // too small for it
  CHECK(d != a);
  pool.free(d);
  pool.release();
  CHECK(g_driver.empty() && pool.cached() == 0);
  return 0;
}

// Read-backs whose sizes wander: once the pool is full, a new size replaces an old one instead of being page-locked every time.
static int wanderingSizes() {
  HostPool pool(HostPoolBackend{mockMalloc, mockFree});
  for (size_t rows = 256; rows <= 3000; rows += 56) {
    std::vector<void *> held;
    for (int i = 0; i < 4; ++i) held.push_back(pool.alloc(rows * 8192));
    for (void *p : held) pool.free(p);
    CHECK(pool.cached() <= HostPool::kMaxCached);
  }
  const int before = g_locks;
  for (int i = 0; i < 100; ++i) {
    void *p = pool.alloc(6500 * 8192);
    CHECK(p != nullptr);
    pool.free(p);
  }
  CHECK(g_locks - before <= 1);
  pool.release();
  CHECK(g_driver.empty());
  return 0;
}

static int bounds() {
  HostPool pool(HostPoolBackend{mockMalloc, mockFree});
  std::vector<void *> held;
  for (int i = 0; i < 4; ++i) { held.push_back(pool.alloc(256 * MiB)); CHECK(held.back() != nullptr); }
  CHECK(pool.alloc(4096) == nullptr);       // kMaxTotal is out
  pool.free(held.back());
  held.pop_back();
  CHECK(pool.cached() == 256 * MiB);
  void *p = pool.alloc(100 * MiB);          // makes room for itself among what is kept
  CHECK(p != nullptr && pool.cached() == 0);
  CHECK(pool.alloc(200 * MiB) == nullptr);
  pool.release();                           // blocks in use are not touched
  CHECK(g_driver.size() == 4);
  pool.free(p);
  for (void *q : held) pool.free(q);
  CHECK(pool.cached() <= HostPool::kMaxCached);
  void *big = pool.alloc(300 * MiB);        // larger than what may be kept
  CHECK(big != nullptr);
  const size_t kept = pool.cached();
  pool.free(big);
  CHECK(pool.cached() == kept);
  g_fail_next = 1;
  CHECK(pool.alloc(700 * MiB) == nullptr);  // the driver's refusal counts nothing
  void *q = pool.alloc(700 * MiB);
  CHECK(q != nullptr);
  pool.free(q);
  pool.release();
  CHECK(g_driver.empty());
  return 0;
}

int main() { return reuse() || wanderingSizes() || bounds(); }
