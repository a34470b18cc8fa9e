// The volumetric shade kernel of the adjoint render's replay (volume.hip launches it).
#include "volume_kernel.h"

namespace lgpu {

void LaunchVolAdjoint(uint32_t blocks, hipStream_t stream, const DevScene *scp, int programs, const RenderParams &rp,
                 PathState ps, SampleState ss, uint32_t n, Queues q, uint32_t *spill, const AdjRefs &ar, const uint32_t *np, BounceSlot *slot) {
  if (programs == kTexPrograms)
    hipLaunchKernelGGL((k_shade_vol<kTexPrograms, kVolAdjoint>), dim3(blocks), dim3(kBlock), 0, stream, scp, rp, ps, ss, n, np, q, spill, ar, slot);
  else if (programs)
    hipLaunchKernelGGL((k_shade_vol<kVmPrograms, kVolAdjoint>), dim3(blocks), dim3(kBlock), 0, stream, scp, rp, ps, ss, n, np, q, spill, ar, slot);
  else
    hipLaunchKernelGGL((k_shade_vol<kNoPrograms, kVolAdjoint>), dim3(blocks), dim3(kBlock), 0, stream, scp, rp, ps, ss, n, np, q, spill, ar, slot);
}

}  // namespace lgpu
