// The part of the HIP runtime that liblambda_gpu.so calls, on host memory: allocations from a budget,
// copies as memcpy, kernels that do nothing. Loaded before the library (RTLD_GLOBAL) it lets the library's
// host code run without a GPU: what it allocates, gives back and copies, and what it does when an
// allocation fails. No result of a kernel can be tested with it.
#include <hip/hip_runtime_api.h>

#include <unistd.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

namespace {
std::mutex mu;
std::map<uintptr_t, size_t> device_mem, pinned_mem;
size_t budget = 4ull << 30, live = 0;
struct Copy {
  uint64_t host, bytes, kind, thread;
};
std::vector<Copy> copies;

void *Take(std::map<uintptr_t, size_t> &m, size_t n) {
  void *p = nullptr;
  if (posix_memalign(&p, 4096, std::max<size_t>(n, 4096))) return nullptr;
  if (n <= (1u << 20)) std::memset(p, 0, n);  // small buffers hold counters the host reads back
  m[reinterpret_cast<uintptr_t>(p)] = n;
  return p;
}
size_t Give(std::map<uintptr_t, size_t> &m, void *p) {
  auto it = m.find(reinterpret_cast<uintptr_t>(p));
  if (it == m.end()) return 0;
  const size_t n = it->second;
  m.erase(it);
  std::free(p);
  return n;
}
bool Holds(const std::map<uintptr_t, size_t> &m, const void *p) {
  auto it = m.upper_bound(reinterpret_cast<uintptr_t>(p));
  if (it == m.begin()) return false;
  --it;
  return reinterpret_cast<uintptr_t>(p) < it->first + it->second;
}
thread_local struct {
  dim3 grid, block;
  size_t shmem;
  hipStream_t stream;
} config;
}  // namespace

extern "C" {
// ---- the test's side
void host_hip_budget(uint64_t bytes) { budget = bytes; }
uint64_t host_hip_live(void) { return live; }
uint64_t host_hip_pinned(void) {
  std::lock_guard<std::mutex> lk(mu);
  uint64_t b = 0;
  for (const auto &x : pinned_mem) b += x.second;
  return b;
}
uint64_t host_hip_copies(Copy *out, uint64_t max) {  // copies since the last call
  std::lock_guard<std::mutex> lk(mu);
  const uint64_t n = copies.size();
  for (uint64_t k = 0; k < n && k < max; ++k) out[k] = copies[k];
  copies.clear();
  return n;
}

// ---- the runtime's side
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipMemGetInfo(size_t *freeB, size_t *totalB) {
  *totalB = budget;
  *freeB = budget - std::min(budget, live);
  return hipSuccess;
}
hipError_t hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  *p = live + n <= budget ? Take(device_mem, n) : nullptr;
  if (!*p) return hipErrorOutOfMemory;
  live += n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  std::lock_guard<std::mutex> lk(mu);
  live -= Give(device_mem, p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  std::lock_guard<std::mutex> lk(mu);
  *p = Take(pinned_mem, n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void *p) {
  std::lock_guard<std::mutex> lk(mu);
  Give(pinned_mem, p);
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
  std::lock_guard<std::mutex> lk(mu);
  std::memset(a, 0, sizeof(*a));
  a->type = Holds(pinned_mem, p) ? hipMemoryTypeHost : Holds(device_mem, p) ? hipMemoryTypeDevice : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipMemcpy(void *dst, const void *src, size_t n, hipMemcpyKind k) {
  std::memcpy(dst, src, n);
  std::lock_guard<std::mutex> lk(mu);
  copies.push_back(Copy{reinterpret_cast<uintptr_t>(k == hipMemcpyHostToDevice ? src : dst), n, (uint64_t)k, (uint64_t)gettid()});
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(dst, src, n, k); }
hipError_t hipMemset(void *p, int v, size_t n) { std::memset(p, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(std::malloc(1)); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = reinterpret_cast<hipEvent_t>(std::malloc(1)); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) {
  static void *scratch = aligned_alloc(4096, 64u << 20);
  *p = scratch;
  return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) { *n = 1; return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shmem, hipStream_t s) {
  config = {grid, block, shmem, s};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shmem, hipStream_t *s) {
  *grid = config.grid;
  *block = config.block;
  *shmem = config.shmem;
  *s = config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
}
