// The volumetric shade kernel of the faithful estimator (volume.hip launches it).
#include "volume_kernel.h"

namespace lgpu {

void LaunchVolFaithful(uint32_t blocks, hipStream_t stream, const DevScene &sc, const RenderParams &rp,
                 PathState ps, SampleState ss, uint32_t n, Queues q, uint32_t *spill, const uint32_t *np, BounceSlot *slot) {
  if (sc.has_programs)
    hipLaunchKernelGGL((k_shade_vol<kVmPrograms, kVolFaithful>), dim3(blocks), dim3(kBlock), 0, stream, sc, rp, ps, ss, n, np, q, spill, AdjRefs{}, slot);
  else
    hipLaunchKernelGGL((k_shade_vol<kNoPrograms, kVolFaithful>), dim3(blocks), dim3(kBlock), 0, stream, sc, rp, ps, ss, n, np, q, spill, AdjRefs{}, slot);
}

}  // namespace lgpu
