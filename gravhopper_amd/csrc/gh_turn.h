// Turns of several wavefronts at data they share: whoever holds turn g waits for it, works on
// the data and passes g + 1 on.  The wait is an acquire and the pass a release, so each turn's
// writes come before the next turn's reads by the memory model.  Plain C++ without hipcc:
// tests/host/turn_check.cpp runs the same turns on threads under ThreadSanitizer.
#pragma once

namespace gh {

constexpr int kTurnWait = __ATOMIC_ACQUIRE;
constexpr int kTurnPass = __ATOMIC_RELEASE;

#ifdef __HIPCC__

__device__ __forceinline__ bool turn_is(const int* turn, int g)
{
    return __hip_atomic_load(turn, kTurnWait, __HIP_MEMORY_SCOPE_WORKGROUP) == g;
}

// Called by a whole wavefront; its lane 0 passes the turn on, after what all its lanes wrote.
// The release makes it wait for those writes, which a relaxed store need not (LDS serves a
// wavefront in order): 1 to 3 % of the FP64 direct sum.
__device__ __forceinline__ void turn_pass(int* turn, int next)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if ((threadIdx.x & 63) == 0)
        __hip_atomic_store(turn, next, kTurnPass, __HIP_MEMORY_SCOPE_WORKGROUP);
}

#else

inline bool turn_is(const int* turn, int g) { return __atomic_load_n(turn, kTurnWait) == g; }

inline void turn_pass(int* turn, int next) { __atomic_store_n(turn, next, kTurnPass); }

#endif

}  // namespace gh
