// Copies of device results to the caller's ordinary host memory.
//
// A copy to ordinary (pageable) memory goes through a staging buffer of the runtime on one CPU
// thread, which also takes the page faults of fresh result arrays, where the link moves 57 GB/s to
// pinned memory.  Large copies are therefore staged here: threads take chunks of the range in
// turn, each copying its chunk from a pinned slot of its own while the other threads' slots are on
// the link, so that faults and memory copies run on several cores.  Not staged / staged, GB/s (MB of 2^20):
//   fresh array      24 MB  10 / 15    48 MB 9.9 / 22    131 MB 10 / 25    375 MB 10 / 33
//   written array    24 MB  18 / 23    48 MB  17 / 26    131 MB 17 / 27    375 MB 17 / 34
// The slots and the threads live for one call.  (The other way the runtime reaches 28 GB/s from
// memory the caller has written, and stays in use.)
#include "sem_device.h"
#include "staged_copy.h"

#include <algorithm>

namespace {

// Slots, one per thread.  Pinned memory costs 0.09 ms a MB in most calls, hardly anything in others or up
// to 6 MB (seen in the calls' times, not explained): with two slots of 2 MB for each of eight threads, 32 MB in
// all, 24 MB took 0.9 to 3.8 ms, against 1.4 (written memory) and 2.5 (fresh) unstaged, 48 MB 1.6 to 4.5
// against 2.9 and 5.1.  Six slots of 1 MB: 24 MB 1.0 to 1.7, 48 MB 1.9 to 2.2; of 512 KB 48 MB in 2.8.  Large
// copies are worth slots of 2 MB: 90 MB 2.6 to 4.5 against 5.4 and 9.2, 375 MB 11.5 ms (1 MB: 13.1).
constexpr int STAGE_THREADS = 6;
constexpr size_t STAGE_CHUNK = (size_t)1 << 20;
constexpr size_t STAGE_LARGE = (size_t)64 << 20;  // from here on 2 * STAGE_CHUNK
// below this the slots and threads (about 0.3 ms) cost what they save
constexpr size_t STAGE_MIN = (size_t)16 << 20;

struct DeviceLink {
  int device;
  char* pinned;
  const char* dev;
  hipStream_t s;
  size_t chunk;
  hipEvent_t ev[STAGE_THREADS];
  char* slot(int w) { return pinned + (size_t)w * chunk; }
  int begin(int w) {
    const int e = hipSetDevice(device);
    return e ? e : (int)hipEventCreateWithFlags(&ev[w], hipEventDisableTiming);
  }
  int fetch(int w, size_t offset, size_t n) {
    const int e = hipMemcpyAsync(slot(w), dev + offset, n, hipMemcpyDeviceToHost, s);
    return e ? e : (int)hipEventRecord(ev[w], s);
  }
  int wait(int w) { return hipEventSynchronize(ev[w]); }
  int end(int w) { return hipEventDestroy(ev[w]); }
};

bool staged_to_host(char* host, const char* dev, size_t bytes, hipStream_t s) {
  DeviceLink link{0, nullptr, dev, s, bytes < STAGE_LARGE ? STAGE_CHUNK : 2 * STAGE_CHUNK, {}};
  HIP_CHECK(hipGetDevice(&link.device));
  if (hipHostMalloc((void**)&link.pinned, STAGE_THREADS * link.chunk, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  HIP_CHECK((hipError_t)staged_copy(host, bytes, link.chunk, STAGE_THREADS, link));
  HIP_CHECK(hipHostFree(link.pinned));
  return true;
}

// c_ij kernels of one element from rows [21][125] to the caller's [125][21], negated, through LDS
__global__ __launch_bounds__(256) void k_cij_point_major(const double* __restrict__ K, double* __restrict__ out) {
  __shared__ double s[2625];
  const size_t b = (size_t)blockIdx.x * 2625;
  for (int i = threadIdx.x; i < 2625; i += 256) s[i] = K[b + i];
  __syncthreads();
  for (int i = threadIdx.x; i < 2625; i += 256) out[b + i] = -s[(i % 21) * 125 + i / 21];
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

void* sem_alloc_part(size_t n, size_t unit_bytes, size_t limit, size_t* units) {
  size_t k = std::min(n, std::max<size_t>(1, limit / unit_bytes));
  void* p = nullptr;
  while (hipMalloc(&p, k * unit_bytes) != hipSuccess) {
    (void)hipGetLastError();
    if (k == 1) SEM_FAIL("no device memory left (%zu bytes needed)", unit_bytes);
    k = (k + 1) / 2;
  }
  *units = k;
  return p;
}

// Kernels are reordered on the device before their copy, a bounded part at a time: a run that fills
// the device still gets its results out.
void sem_cij_to_host(const SemMesh* m, const double* K, size_t n, double* host) {
  constexpr size_t EL = 2625;
  size_t most = 0;
  double* tmp = (double*)sem_alloc_part(n, EL * sizeof(double), m->readout_bytes, &most);
  for (size_t e = 0; e < n; e += most) {
    const size_t k = std::min(most, n - e);
    hipLaunchKernelGGL(k_cij_point_major, dim3((unsigned)k), dim3(256), 0, m->stream, K + e * EL, tmp);
    HIP_CHECK(hipGetLastError());
    sem_to_host(host + e * EL, tmp, k * EL * sizeof(double), m->stream);
  }
  dev_free(tmp);
}
