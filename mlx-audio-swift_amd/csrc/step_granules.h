// step_granules.h - device code that the decode steps in one launch share (lm_step.hip, whisper_step.hip): values from block to block as granules, waits that end
#pragma once
#include "lm_step.h"

typedef unsigned long long u64;
// a granule: two bfloat16 values and the tag that says whose they are - one store, no flag, nothing to wait for
__device__ __forceinline__ void granule(unsigned char* p, uint32_t v, unsigned tag) { __hip_atomic_store(reinterpret_cast<u64*>(p), (u64)v | (u64)tag << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float bf_lo(uint32_t v) { return bf16_to_f32((bf16_t)(v & 0xffffu)); }
__device__ __forceinline__ float bf_hi(uint32_t v) { return bf16_to_f32((bf16_t)(v >> 16)); }
__device__ __forceinline__ void bar() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The kernel's arguments, read again (scalar loads) from here on: kept in registers over the layer loop they are more than there are.
template <class P> __device__ __forceinline__ const P& step_args() {
    typedef __attribute__((address_space(4))) const P* ArgPtr;
    ArgPtr a = (ArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return *(const P*)a;
}
// A poll in vain, t0 the time of the first (0: this one): false where some block has run out of time, or this one now has, and says so
template <class P> __device__ __forceinline__ bool more_time(u64& t0, int lane) {
    const P& p = step_args<P>();
    const u64 now = wall_clock64();
    if (t0 == 0) t0 = now;
    if (__builtin_amdgcn_readfirstlane(__hip_atomic_load(p.fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0) return false;
    if (now - t0 < p.limit) return true;
    if (lane == 0) {
        __hip_atomic_store(p.sync + SYNC_LATE, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(p.fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return false;
}
