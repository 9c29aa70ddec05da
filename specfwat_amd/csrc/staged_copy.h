// A copy through staging slots by several threads, whatever the link: sem_to_host's threads
// (transfer.hip), host code only.
#pragma once
#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

// Copies bytes to host by at most `threads` workers, chunk bytes at a time, each worker through a slot of
// its own: the link serves the others while one copies from its slot.  Link (calls return 0 or an error):
//   begin(w), end(w)         worker w starts, on its own thread, and ends (after a begin that succeeded)
//   fetch(w, offset, n)      starts bringing n bytes from offset into the slot of w
//   wait(w), slot(w)         waits for the last fetch into the slot; the slot's memory
// Returns the first error, after which no worker starts anything more, once all workers have
// ended: the caller alone decides what an error does to the process.
template <class Link>
int staged_copy(char* host, size_t bytes, size_t chunk, int threads, Link& link) {
  const size_t chunks = (bytes + chunk - 1) / chunk;
  std::atomic<size_t> next{0};
  std::atomic<int> ids{0}, error{0};
  const auto ok = [&](int e) {
    int none = 0;
    if (e) error.compare_exchange_strong(none, e);
    return e == 0;
  };
  const auto work = [&] {
    const int w = ids.fetch_add(1);
    if (!ok(link.begin(w))) return;
    for (size_t c = next.fetch_add(1); c < chunks && !error.load(); c = next.fetch_add(1)) {
      const size_t n = std::min(chunk, bytes - c * chunk);
      if (!ok(link.fetch(w, c * chunk, n)) || !ok(link.wait(w))) break;
      std::memcpy(host + c * chunk, link.slot(w), n);
    }
    ok(link.end(w));
  };
  std::vector<std::thread> team;
  const int others = (int)std::min<size_t>((size_t)threads, chunks) - 1;
  try {
    team.reserve(others);
    for (int t = 0; t < others; ++t) team.emplace_back(work);
  } catch (const std::exception&) {  // fewer threads: the ones there are take all chunks
  }
  work();
  for (auto& t : team) t.join();
  return error.load();
}
