// Copies of device results to the caller's ordinary host memory.
//
// A copy to ordinary (pageable) memory goes through a staging buffer of the runtime on one CPU
// thread, which also takes the page faults of fresh result arrays: 131 MB of kernels took 12 to
// 22 ms (6 to 11 GB/s), where the link moves 57 GB/s to pinned memory.  Large copies are
// therefore staged here: threads take chunks of the range in turn, each copying its chunk from
// a pinned slot of its own while the other threads' slots are on the link, so that faults and
// memory copies run on several cores.  The slots and the threads live for one call.  (The other way the
// runtime reaches 28 GB/s from memory the caller has written, and stays in use.)
#include "sem_device.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>
#include <vector>

namespace {

constexpr size_t STAGE_CHUNK = (size_t)2 << 20;
constexpr int STAGE_THREADS = 8;
// below this the slots and threads (about 0.5 ms) cost more than they save
constexpr size_t STAGE_MIN = (size_t)16 << 20;

bool staged_to_host(char* host, const char* dev, size_t bytes, hipStream_t s) {
  const size_t chunks = (bytes + STAGE_CHUNK - 1) / STAGE_CHUNK;
  int device = 0;
  HIP_CHECK(hipGetDevice(&device));
  char* pinned = nullptr;
  if (hipHostMalloc((void**)&pinned, 2 * STAGE_THREADS * STAGE_CHUNK, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  std::atomic<size_t> next{0};
  std::atomic<int> ids{0};
  // two slots per thread: one on the link while the other is copied from
  const auto work = [&] {
    HIP_CHECK(hipSetDevice(device));
    char* slot = pinned + 2 * STAGE_CHUNK * (size_t)ids.fetch_add(1);
    hipEvent_t ev[2];
    for (auto& e : ev) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    size_t held[2] = {chunks, chunks};  // the chunk of each slot, chunks: none
    const auto size_of = [&](size_t c) { return std::min(STAGE_CHUNK, bytes - c * STAGE_CHUNK); };
    const auto hand_over = [&](int b) {
      if (held[b] == chunks) return;
      HIP_CHECK(hipEventSynchronize(ev[b]));
      std::memcpy(host + held[b] * STAGE_CHUNK, slot + b * STAGE_CHUNK, size_of(held[b]));
      held[b] = chunks;
    };
    int b = 0;
    for (size_t c = next.fetch_add(1); c < chunks; c = next.fetch_add(1), b ^= 1) {
      hand_over(b);
      HIP_CHECK(hipMemcpyAsync(slot + b * STAGE_CHUNK, dev + c * STAGE_CHUNK, size_of(c), hipMemcpyDeviceToHost, s));
      HIP_CHECK(hipEventRecord(ev[b], s));
      held[b] = c;
    }
    hand_over(b);
    hand_over(b ^ 1);
    for (auto& e : ev) HIP_CHECK(hipEventDestroy(e));
  };
  std::vector<std::thread> team;
  const int others = (int)std::min<size_t>(STAGE_THREADS, chunks) - 1;
  try {
    team.reserve(others);
    for (int t = 0; t < others; ++t) team.emplace_back(work);
  } catch (const std::exception&) {  // fewer threads: the ones there are take all chunks
  }
  work();
  for (auto& t : team) t.join();
  HIP_CHECK(hipHostFree(pinned));
  return true;
}

bool pageable(const void* host) {
  hipPointerAttribute_t at;
  if (hipPointerGetAttributes(&at, host) == hipSuccess) return at.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

}  // namespace

// The copy is complete on return; work queued on s before runs before it.
void sem_to_host(void* host, const void* dev, size_t bytes, hipStream_t s) {
  if (bytes == 0) return;
  if (bytes >= STAGE_MIN && pageable(host) && staged_to_host((char*)host, (const char*)dev, bytes, s)) return;
  HIP_CHECK(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
}
