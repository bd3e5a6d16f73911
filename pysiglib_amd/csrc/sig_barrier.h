// Barrier of a block that exchanges data through LDS only.
#pragma once
#include <hip/hip_runtime.h>

namespace sigamd {

// __syncthreads also waits for a wave's global loads and stores, which would end here what is meant to be in flight across it.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);     // own LDS operations have completed (vmcnt and expcnt at their maxima)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

}  // namespace sigamd
