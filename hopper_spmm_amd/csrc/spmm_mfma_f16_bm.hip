// Instantiations of the MFMA kernel: element type f16, single windows, tiles as bitmap + stored elements.
#include <hip/hip_runtime.h>
#include "spmm_mfma_kernel.hpp"

namespace hspmm {

hipError_t launch_mfma_f16_bm(const KernelArgs &ka, int V, int prefetch, bool narrow, int waves_per_group, hipStream_t s,
                            hipEvent_t mid)
{
    if (V == 4) return launch_tt<Fp16TileDWB<4, false>>(ka, prefetch, narrow, waves_per_group, s, mid);
    if (V == 2) return launch_tt<Fp16TileDWB<2, false>>(ka, prefetch, narrow, waves_per_group, s, mid);
    return hipErrorInvalidValue;
}

hipError_t launch_mfma_f16_scheduled(const KernelArgs &ka, int waves_per_group, hipStream_t s, hipEvent_t mid)
{
    return launch_default<Scheduled<Fp16TileDWB<2, false>>>(ka, waves_per_group, s, mid);
}

}  // namespace hspmm
