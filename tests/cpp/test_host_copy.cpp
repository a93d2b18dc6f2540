// Shared host copies: values at the edges of the chunks, several callers at once, a process that may start no thread, and a forked
// child, which has none of its parent's helpers.
// Build: g++ -std=c++17 -pthread -I tt-mlir_amd/runtime tests/cpp/test_host_copy.cpp -o <exe>; exit status 0 = all checks passed.
#include <sys/resource.h>
#include <sys/wait.h>
#include <unistd.h>

#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "host_copy.h"

using tt::runtime::HostCopy;

#define CHECK(cond)                                                          \
  do {                                                                       \
    if (!(cond)) { std::fprintf(stderr, "%s:%d: CHECK(%s) failed\n", __FILE__, __LINE__, #cond); return 1; } \
  } while (0)

static int copies(size_t bytes, unsigned seed) {
  std::vector<unsigned char> src(bytes + 2), dst(bytes + 2, 7);
  for (size_t i = 0; i < src.size(); ++i) src[i] = static_cast<unsigned char>((i * 2654435761u + seed) >> 13);
  HostCopy::run(dst.data() + 1, src.data() + 1, bytes);
  CHECK(dst.front() == 7 && dst.back() == 7);
  CHECK(std::equal(dst.begin() + 1, dst.end() - 1, src.begin() + 1));
  return 0;
}

static int sizes() {
  for (size_t bytes : {size_t(0), size_t(1), HostCopy::kShareFrom - 1, HostCopy::kShareFrom, HostCopy::kShareFrom + 1,
                       HostCopy::kShareFrom + HostCopy::kChunk - 1, size_t(16) << 20})
    if (copies(bytes, 1)) return 1;
  return 0;
}

static int manyCallers() {
  std::vector<std::thread> ts;
  std::vector<int> bad(6, 0);
  for (int t = 0; t < 6; ++t)
    ts.emplace_back([t, &bad] {
      for (int k = 0; k < 20; ++k) bad[t] |= copies(HostCopy::kShareFrom + 100000u * t + k, t * 100 + k);
    });
  for (auto &t : ts) t.join();
  for (int b : bad) CHECK(b == 0);
  return 0;
}

// f in a child process that is killed after ten seconds
template <typename F>
static int inChild(F f) {
  const pid_t pid = fork();
  if (pid == 0) {
    alarm(10);
    _exit(f());
  }
  int status = 0;
  CHECK(waitpid(pid, &status, 0) == pid);
  CHECK(WIFEXITED(status) && WEXITSTATUS(status) == 0);
  return 0;
}

static int withoutThreads() {   // no room for another stack
  long pages = 0;
  FILE *f = std::fopen("/proc/self/statm", "r");
  CHECK(f && std::fscanf(f, "%ld", &pages) == 1);
  std::fclose(f);
  const rlim_t room = static_cast<rlim_t>(pages) * static_cast<rlim_t>(sysconf(_SC_PAGESIZE)) + (rlim_t(13) << 20);
  const rlimit lim = {room, room};
  CHECK(setrlimit(RLIMIT_AS, &lim) == 0);
  for (int k = 0; k < 50; ++k)
    if (copies(HostCopy::kShareFrom + k, k)) return 1;
  return 0;
}

int main() {
  if (inChild(withoutThreads)) return 1;   // before this process has helpers
  if (sizes() || manyCallers()) return 1;
  for (int k = 0; k < 20; ++k)
    if (inChild(sizes)) return 1;
  std::thread busy([] { for (int k = 0; k < 200; ++k) (void)copies(size_t(4) << 20, k); });
  int bad = 0;
  for (int k = 0; k < 20 && !bad; ++k) bad = inChild(sizes);   // forked while another thread shares its copies out
  busy.join();
  return bad;
}
