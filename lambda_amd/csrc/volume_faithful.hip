// The volumetric shade kernel of the faithful estimator (volume.hip launches it).
#include "volume_kernel.h"

namespace lgpu {

void LaunchVolFaithful(uint32_t blocks, hipStream_t stream, const DevScene *scp, int programs, const RenderParams &rp,
                 PathState ps, SampleState ss, uint32_t n, Queues q, uint32_t *spill, const uint32_t *np, BounceSlot *slot) {
  if (programs)
    hipLaunchKernelGGL((k_shade_vol<kVmPrograms, kVolFaithful>), dim3(blocks), dim3(kBlock), 0, stream, scp, rp, ps, ss, n, np, q, spill, AdjRefs{}, slot);
  else
    hipLaunchKernelGGL((k_shade_vol<kNoPrograms, kVolFaithful>), dim3(blocks), dim3(kBlock), 0, stream, scp, rp, ps, ss, n, np, q, spill, AdjRefs{}, slot);
}

}  // namespace lgpu
