// Barrier between the workgroups (members) that share a pair or a sequence:
// an arrival counter per pair, cleared before the launch, and a bounded wait.
#pragma once
#include <hip/hip_runtime.h>

#define LCG_WAIT_EXPIRED (1 << 30)  // in the counter; arrivals stay far below

// Arrival and wait for `target` arrivals in at most `polls` polls, -1: none
// (one thread of each member); false: this wait or an earlier one of any
// member expired.  An expired wait stays in the counter, so that no later one
// waits for members that are behind, and so that these learn of it when they
// come (what they then write, others may have read before).
__device__ __forceinline__ bool arrive_and_wait(int *counter, int target, int polls) {
    int seen = atomicAdd(counter, 1) + 1;
    for (int spin = 0; polls < 0 || seen < target; ++spin) {
        if (spin > polls) {
            atomicOr(counter, LCG_WAIT_EXPIRED);
            return false;
        }
        __builtin_amdgcn_s_sleep(2);
        seen = atomicAdd(counter, 0);
    }
    return seen < LCG_WAIT_EXPIRED;
}

// What every member wrote to global memory before it, every member reads after
// it.  A member's waves run on one CU: each waits until its own stores are in
// the L2 (vmcnt(0); neither s_barrier nor a fence of workgroup scope waits for
// them), and only then does one wave write the L2 back, arrive and, once all
// have arrived, drop what the CU's L1 and the L2 hold of other XCDs' memory: a
// write-back and an invalidation per member, not per wave (a barrier of 16
// waves 30 us with one per wave, 7 us so).
// `expired` is called by one thread where arrive_and_wait returns false.
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
