// Runs staged_copy over a link of plain memory: prints "ok" when every copy is whole and every
// failing call comes back as its error with all workers ended.
#include "staged_copy.h"

#include <chrono>
#include <cstdio>
#include <random>

struct MemoryLink {
  const std::vector<char>& src;
  size_t chunk;
  int fail_at = -1;  // the call (counted over all workers) that fails
  std::atomic<int> calls{0}, inside{0}, begun{0}, ended{0};
  std::vector<char> slots;
  struct Fetch { size_t offset, n; } last[8];
  MemoryLink(const std::vector<char>& s, size_t c) : src(s), chunk(c), slots(8 * c) {}
  int call() {
    std::this_thread::sleep_for(std::chrono::microseconds(calls.load() % 7));
    return calls.fetch_add(1) == fail_at ? 77 : 0;
  }
  char* slot(int w) { return slots.data() + (size_t)w * chunk; }
  int begin(int) {
    const int e = call();
    if (!e) ++inside, ++begun;
    return e;
  }
  int fetch(int w, size_t offset, size_t n) {
    last[w] = {offset, n};
    return call();
  }
  int wait(int w) {  // the data arrive here at the latest
    const int e = call();
    if (!e) std::memcpy(slot(w), src.data() + last[w].offset, last[w].n);
    return e;
  }
  int end(int) {
    --inside, ++ended;
    return call();
  }
};

int main() {
  std::mt19937 rng(3);
  const size_t chunk = 64;
  for (size_t bytes : {1, 63, 64, 65, 127, 500, 8 * 64, 8 * 64 + 1, 5000, 6399, 6400}) {
    std::vector<char> src(bytes);
    for (auto& x : src) x = (char)rng();
    int total = 0;
    for (int fail = -1; fail <= total; ++fail) {
      MemoryLink link(src, chunk);
      link.fail_at = fail < 0 ? -1 : fail;
      std::vector<char> host(bytes + 1, 0);
      const int e = staged_copy(host.data(), bytes, chunk, 8, link);
      const bool hit = fail >= 0 && link.calls > fail;
      if (e != (hit ? 77 : 0) || link.inside != 0 || link.begun != link.ended || host[bytes] != 0) {
        std::printf("bytes %zu fail %d: error %d, %d workers inside\n", bytes, fail, e, link.inside.load());
        return 1;
      }
      if (e == 0 && std::memcmp(host.data(), src.data(), bytes) != 0) {
        std::printf("bytes %zu: copy differs\n", bytes);
        return 1;
      }
      if (fail < 0) total = link.calls;
    }
  }
  std::puts("ok");
}
