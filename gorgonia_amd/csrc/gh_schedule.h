// The order of a step's loads and matrix instructions.
#pragma once

// A loop whose step loads the next step's operands and multiplies the present ones: left alone the compiler puts the loads behind
// the matrix instructions, where it needs fewer registers, and waits for them there.  Kept in front of them in one go
// (sched_barrier) they keep the wavefront, and through the unit that works out the lanes' addresses all others of the compute unit,
// from its matrix instructions: float32 793 x 1468, K = 3357 on k_gemm_direct takes 87.2 us as the compiler has it, 140 with
// the loads in front, 69.6 with each behind a few matrix instructions.

// One of kLoads loads behind every few of kMacs matrix instructions: those that stand with them in front of the call, in the
// order in which they stand there.
template <int kLoads, int kMacs, int I = 0>
__device__ __forceinline__ void gh_spread_loads() {
  if constexpr (I < kLoads) {
    __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);   // a load
    constexpr int n = (I + 1) * kMacs / kLoads - I * kMacs / kLoads;
    if constexpr (n > 0) __builtin_amdgcn_sched_group_barrier(0x008, n, 0);   // matrix instructions
    gh_spread_loads<kLoads, kMacs, I + 1>();
  }
}
