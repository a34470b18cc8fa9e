// Copies between device memory and a caller's (pageable) arrays. The runtime's own copy of pageable
// memory moves it through one staging buffer on one thread: 50 MB of film into fresh pages took 6 ms,
// most of it page faults and memcpy. Here the transfer runs in chunks through pinned buffers kept on the
// device object, and a few threads copy finished chunks (and fault the pages in) while later ones are
// on the bus. The calling thread is one of them and starts at once; it wakes a helper only for a chunk
// beyond its own buffers, and takes back a helper that has not woken by the time no chunk is left. A read
// that woke all six threads and waited for them took 116 us at 1.1 MiB and 160 at 2 MiB, where the runtime
// takes 95 and 133 and this 90 and 121. Small copies go straight to the runtime.
// Ray batch of 1,000,003 (intersect and occluded, 84 MB of copies) 5.6 -> 3.6 ms, 1080p film read of the
// many-light render 79.6 -> 75.6 ms for the whole pass.
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <thread>

#include "host.h"

namespace lgpu {

namespace {

constexpr size_t kChunk = 1u << 20;    // bytes per transfer
constexpr int kCopyThreads = 6;        // the caller and five helpers
constexpr int kOwn = 2;                // pinned buffers of a thread: one is copied while the other is on the bus
constexpr int kChunks = kOwn * kCopyThreads;  // 12 MiB per device object
// Copies up to this size (one chunk) are the runtime's. In place, as it copies larger arrays to the device, it is
// faster (film writes of 2, 8 and 24 MiB 97, 309 and 824 us, chunks 108, 415 and 1042), but the pages it has
// locked cost later: one in three first passes on new films of 8 MiB then took 3 to 5 ms instead of 0.6.
constexpr size_t kDirect = 1u << 20;

struct HostCopier {
  uint8_t *pinned = nullptr;
  hipEvent_t done[kChunks] = {};
  std::vector<std::thread> threads;
  std::mutex mu;
  std::condition_variable wake, idle;
  bool stop = false;
  int tickets = 0;  // helpers the current job still wants
  int busy = 0;     // helpers at work on it; the fields below describe it
  int device = 0;
  hipStream_t stream = nullptr;
  uint8_t *host = nullptr, *dev = nullptr;
  size_t bytes = 0;
  bool toHost = true;
  std::atomic<size_t> next{0};
  std::atomic<int> error{0};

  ~HostCopier() {
    {
      std::lock_guard<std::mutex> lk(mu);
      stop = true;
    }
    wake.notify_all();
    for (std::thread &t : threads) t.join();
    for (hipEvent_t e : done)
      if (e) (void)hipEventDestroy(e);
    if (pinned) (void)hipHostFree(pinned);
  }
  // Each thread owns kOwn buffers and takes the next chunk of the job for each.
  void Work(int id) {
    const size_t count = (bytes + kChunk - 1) / kChunk;
    size_t at[kOwn];
    bool full[kOwn] = {};
    (void)hipSetDevice(device);
    auto finish = [&](int k) {
      const int b = id * kOwn + k;
      hipError_t e = hipEventSynchronize(done[b]);
      if (e != hipSuccess) error = (int)e;
      else if (toHost) std::memcpy(host + at[k], pinned + b * kChunk, std::min(kChunk, bytes - at[k]));
      full[k] = false;
    };
    for (int k = 0;; k = (k + 1) % kOwn) {
      if (full[k]) finish(k);
      const size_t c = next.fetch_add(1);
      if (c >= count || error) break;
      const int b = id * kOwn + k;
      const size_t off = c * kChunk, n = std::min(kChunk, bytes - off);
      hipError_t e;
      if (toHost) {
        e = hipMemcpyAsync(pinned + b * kChunk, dev + off, n, hipMemcpyDeviceToHost, stream);
      } else {
        std::memcpy(pinned + b * kChunk, host + off, n);
        e = hipMemcpyAsync(dev + off, pinned + b * kChunk, n, hipMemcpyHostToDevice, stream);
      }
      if (e == hipSuccess) e = hipEventRecord(done[b], stream);
      if (e != hipSuccess) {
        error = (int)e;
        break;
      }
      at[k] = off;
      full[k] = true;
    }
    for (int k = 0; k < kOwn; ++k)
      if (full[k]) finish(k);
  }
  void Loop(int id) {
    std::unique_lock<std::mutex> lk(mu);
    for (;;) {
      wake.wait(lk, [&] { return stop || tickets > 0; });
      if (stop) return;
      --tickets;
      ++busy;
      lk.unlock();
      Work(id);
      lk.lock();
      if (--busy == 0) idle.notify_all();
    }
  }
  // False when a buffer, event or thread cannot be had (the caller then copies through the runtime).
  bool Start() {
    if (!threads.empty()) return true;
    if (!pinned && hipHostMalloc((void **)&pinned, kChunk * kChunks, hipHostMallocDefault) != hipSuccess) pinned = nullptr;
    for (hipEvent_t &e : done)
      if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) e = nullptr;
    (void)hipGetLastError();
    if (!pinned) return false;
    for (hipEvent_t e : done)
      if (!e) return false;
    try {
      for (int k = 1; k < kCopyThreads; ++k) threads.emplace_back([this, k] { Loop(k); });
    } catch (...) {  // fewer threads than asked for: give the started ones back
      {
        std::lock_guard<std::mutex> lk(mu);
        stop = true;
      }
      wake.notify_all();
      for (std::thread &t : threads) t.join();
      threads.clear();
      stop = false;
      return false;
    }
    return true;
  }
  hipError_t Run(lgpu_device d, void *h, void *p, size_t n, bool down) {
    const size_t chunks = (n + kChunk - 1) / kChunk;
    std::unique_lock<std::mutex> lk(mu);
    device = d->device;
    stream = d->stream;
    host = static_cast<uint8_t *>(h);
    dev = static_cast<uint8_t *>(p);
    bytes = n;
    toHost = down;
    next = 0;
    error = 0;
    const int helpers = (int)std::min<size_t>(kCopyThreads - 1, chunks > kOwn ? chunks - kOwn : 0);
    tickets = helpers;
    lk.unlock();
    for (int k = 0; k < helpers; ++k) wake.notify_one();
    Work(0);
    lk.lock();
    tickets = 0;
    idle.wait(lk, [&] { return busy == 0; });
    return (hipError_t)error.load();
  }
};

// Memory that the runtime does not know: neither page-locked (the bus reaches it without a staging copy:
// 3 MiB read in 64 us, 160 through the chunks) nor a device's, which a caller may pass too.
bool Pageable(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
  (void)hipGetLastError();
  return true;
}

hipError_t Copy(lgpu_device d, void *host, void *dev, size_t n, bool down) {
  if (!n) return hipSuccess;
  if (n > kDirect && Pageable(host)) {
    if (!d->copier) {
      try {
        d->copier = new HostCopier();
        d->copier_free = [](void *p) { delete static_cast<HostCopier *>(p); };
      } catch (...) {
        d->copier = nullptr;
      }
    }
    HostCopier *c = static_cast<HostCopier *>(d->copier);
    if (c && c->Start()) return c->Run(d, host, dev, n, down);
  }
  const hipError_t e = down ? hipMemcpyAsync(host, dev, n, hipMemcpyDeviceToHost, d->stream)
                            : hipMemcpyAsync(dev, host, n, hipMemcpyHostToDevice, d->stream);
  return e == hipSuccess ? hipStreamSynchronize(d->stream) : e;
}

}  // namespace

hipError_t CopyToHost(lgpu_device d, void *host, const void *dev, size_t n) {
  return Copy(d, host, const_cast<void *>(dev), n, true);
}
hipError_t CopyToDevice(lgpu_device d, void *dev, const void *host, size_t n) {
  return Copy(d, const_cast<void *>(host), dev, n, false);
}

}  // namespace lgpu
