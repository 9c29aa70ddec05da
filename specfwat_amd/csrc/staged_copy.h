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

// Copies bytes to host by at most `threads` workers, chunk bytes at a time, each worker with two slots:
// one on the link while the other is copied from.  Link (calls return 0 or an error):
//   begin(w), end(w)             worker w starts, on its own thread, and ends (after a begin that succeeded)
//   fetch(w, b, offset, n)       starts bringing n bytes from offset into slot b of w
//   wait(w, b), slot(w, b)       waits for the last fetch into that slot; the slot's memory
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
    size_t held[2] = {chunks, chunks};  // the chunk of each slot, chunks: none
    const auto size_of = [&](size_t c) { return std::min(chunk, bytes - c * chunk); };
    const auto hand_over = [&](int b) {
      if (held[b] == chunks) return true;
      if (error.load() || !ok(link.wait(w, b))) return false;
      std::memcpy(host + held[b] * chunk, link.slot(w, b), size_of(held[b]));
      held[b] = chunks;
      return true;
    };
    int b = 0;
    bool going = true;
    for (size_t c = next.fetch_add(1); going && c < chunks; c = next.fetch_add(1), b ^= 1) {
      going = hand_over(b) && ok(link.fetch(w, b, c * chunk, size_of(c)));
      if (going) held[b] = c;
    }
    if (going && hand_over(b)) hand_over(b ^ 1);
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
