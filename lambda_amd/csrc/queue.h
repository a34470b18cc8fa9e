// Queue pushes of the shading kernels. Slots are handed out per block: a device-scope atomic on one
// counter serialises across the whole GPU (about 11 ns each on MI355X, measured), so one per block
// instead of one per wave cuts that cost fourfold. A thread keeps its extension ray in registers
// until the block's allocation.
#pragma once
#include "lgpu_internal.h"
#include "trace.h"

namespace lgpu {

// Device clock of a stage's start (BounceSlot), written by its first block; nothing without a slot.
__device__ inline void Stamp(unsigned long long *t) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *t = wall_clock64();
}
// Copies a bounce's slot to pinned host memory; called by the first thread of the bounce's last kernel.
// The host reads it after an event that follows the kernel.
__device__ inline void Publish(const BounceSlot *slot, BounceSlot *host) {
  host->next = slot->next;
  host->shadow = slot->shadow;
  host->extend = slot->extend;
  host->infer = slot->infer;
  host->shade = slot->shade;
  host->shadows = slot->shadows;
}

struct ExtPush {
  float4 o, d, beta, mis, pp, pn;
  uint4 ids, aux;
};
__device__ inline void WriteExt(const PathState &next, uint32_t j, const ExtPush &e) {
  next.ray_o[j] = e.o;
  next.ray_d[j] = e.d;
  next.beta[j] = e.beta;
  next.ids[j] = e.ids;
  next.aux[j] = e.aux;
  next.mis[j] = e.mis;
  next.prev_p[j] = e.pp;
  next.prev_n[j] = e.pn;
}
// Appends the block's extension rays; every thread of the block calls it (barriers inside).
// lds: kBlock / 64 + 1 words.
__device__ inline void BlockPushExt(const PathState &next, uint32_t *counter, bool push, const ExtPush &e, uint32_t *lds) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint64_t m = __ballot(push);
  if (lane == 0) lds[wv] = (uint32_t)__popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t total = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
      const uint32_t c = lds[w];
      lds[w] = total;
      total += c;
    }
    lds[kBlock / 64] = total ? atomicAdd(counter, total) : 0u;
  }
  __syncthreads();
  if (push) WriteExt(next, lds[kBlock / 64] + lds[wv] + (uint32_t)__popcll(m & ((1ull << lane) - 1ull)), e);
}

}  // namespace lgpu
