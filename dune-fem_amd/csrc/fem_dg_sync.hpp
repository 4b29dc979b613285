// LDS ordering inside a workgroup whose element groups are single wavefronts
// or whole workgroups (shared by the DG kernels).
#pragma once

#include <hip/hip_runtime.h>

namespace femamd {

// Orders LDS accesses between the lanes of one wavefront.  LDS instructions of
// a wavefront execute in issue order, so only the compiler must be kept from
// moving memory operations across this point; no s_barrier and no wait on
// outstanding global loads is needed.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the exchange barrier of a group of G lanes: a wavefront fence for one
// wavefront, the workgroup barrier for more (the group is then the workgroup)
template <int G>
__device__ __forceinline__ void lds_sync()
{
    if constexpr (G > 64) __syncthreads();
    else wave_lds_sync();
}

}  // namespace femamd
