// Barrier between the workgroups (members) that share a pair or a sequence:
// an arrival counter per pair, cleared before the launch, and a bounded wait.
#pragma once
#include <hip/hip_runtime.h>

// Arrival and wait for `target` arrivals in at most `polls` polls (one thread
// of each member); false: the wait expired.
__device__ __forceinline__ bool arrive_and_wait(int *counter, int target, int polls) {
    atomicAdd(counter, 1);
    for (int spin = 0; polls < 0 || atomicAdd(counter, 0) < target; ++spin) {
        if (spin > polls) return false;
        __builtin_amdgcn_s_sleep(2);
    }
    return true;
}

// What every member wrote to global memory before it, every member reads after
// it.  A member's waves run on one CU: each waits until its own stores are in
// the L2 (vmcnt(0); neither s_barrier nor a fence of workgroup scope waits for
// them), and only then does one wave write the L2 back, arrive and, once all
// have arrived, drop what the CU's L1 and the L2 hold of other XCDs' memory: a
// write-back and an invalidation per member, not per wave.  With a write-back
// per wave a diagonal of lcg_fold_seqs takes 30 us, so 7.
// `expired` is called by one thread if the wait expired.
template <class Expired>
__device__ __forceinline__ void member_barrier(int *counter, int target, int polls, Expired expired) {
    __threadfence_block();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        if (!arrive_and_wait(counter, target, polls)) expired();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }
    __syncthreads();
}
