// Copies between the caller's ordinary host memory and the device.
//
// A copy of ordinary (pageable) memory goes through a staging buffer of the runtime on one CPU
// thread: 131 MB of kernels into fresh pages took 12 to 22 ms (6 to 11 GB/s, the page faults
// among them) and 4.6 ms the other way, where the link moves 57 GB/s from pinned memory.  Large
// copies are therefore staged here: threads take chunks of the range in turn, each copying its
// chunk between the caller's memory and a pinned slot of its own while the other threads' slots
// are on the link, so that faults and memory copies run on several cores.  The slots and the
// threads live for one call.
#include "sem_device.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <system_error>
#include <thread>

namespace {

constexpr size_t STAGE_CHUNK = (size_t)2 << 20;
constexpr int STAGE_THREADS = 8;
// below this the slots and threads (about 0.5 ms) cost more than they save
constexpr size_t STAGE_MIN = (size_t)16 << 20;

bool staged_copy(char* host, char* dev, size_t bytes, hipStream_t s, bool to_device) {
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
  // two slots per thread: one on the link while the other is copied to or from
  const auto work = [&] {
    HIP_CHECK(hipSetDevice(device));
    char* slot = pinned + 2 * STAGE_CHUNK * (size_t)ids.fetch_add(1);
    hipEvent_t ev[2];
    for (auto& e : ev) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    size_t held[2];  // the chunk of each slot on the link, chunks: none
    held[0] = held[1] = chunks;
    const auto size_of = [&](size_t c) { return std::min(STAGE_CHUNK, bytes - c * STAGE_CHUNK); };
    const auto finish = [&](int b) {  // slot b's copy is complete; to the host: hand its chunk over
      if (held[b] == chunks) return;
      HIP_CHECK(hipEventSynchronize(ev[b]));
      if (!to_device) std::memcpy(host + held[b] * STAGE_CHUNK, slot + b * STAGE_CHUNK, size_of(held[b]));
      held[b] = chunks;
    };
    int b = 0;
    for (size_t c = next.fetch_add(1); c < chunks; c = next.fetch_add(1), b ^= 1) {
      finish(b);
      char* p = slot + b * STAGE_CHUNK;
      if (to_device) {
        std::memcpy(p, host + c * STAGE_CHUNK, size_of(c));
        HIP_CHECK(hipMemcpyAsync(dev + c * STAGE_CHUNK, p, size_of(c), hipMemcpyHostToDevice, s));
      } else {
        HIP_CHECK(hipMemcpyAsync(p, dev + c * STAGE_CHUNK, size_of(c), hipMemcpyDeviceToHost, s));
      }
      HIP_CHECK(hipEventRecord(ev[b], s));
      held[b] = c;
    }
    finish(b);
    finish(b ^ 1);
    for (auto& e : ev) HIP_CHECK(hipEventDestroy(e));
  };
  std::vector<std::thread> team;
  const int others = (int)std::min<size_t>(STAGE_THREADS, chunks) - 1;
  try {
    team.reserve(others);
    for (int t = 0; t < others; ++t) team.emplace_back(work);
  } catch (const std::system_error&) {  // fewer threads: the ones there are take all chunks
  }
  work();
  for (auto& t : team) t.join();
  HIP_CHECK(hipHostFree(pinned));
  return true;
}

}  // namespace

// A large copy is complete on return, a small one ordered on s as hipMemcpyAsync orders it.
void sem_to_device(void* dev, const void* host, size_t bytes, hipStream_t s) {
  if (bytes == 0) return;
  if (bytes >= STAGE_MIN && staged_copy((char*)const_cast<void*>(host), (char*)dev, bytes, s, true)) return;
  HIP_CHECK(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, s));
}

// The copy is complete on return.
void sem_to_host(void* host, const void* dev, size_t bytes, hipStream_t s) {
  if (bytes == 0) return;
  if (bytes >= STAGE_MIN && staged_copy((char*)host, (char*)const_cast<void*>(dev), bytes, s, false)) return;
  HIP_CHECK(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
}
