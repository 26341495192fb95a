// Device stores that the host sees in coherent pinned memory while the kernel
// still runs: each goes through the caches whole.  host_stores_wait() returns
// when those of the wavefront have arrived, so that a store after it (and,
// across a workgroup barrier, another wavefront's) tells the host that they
// have.  A system-scope fence in its place also writes back what the L2 holds:
// 12.7 against 8.4 us for a reduce of N = 10,000, P = 2, and 22 against 14 at N
// = 6,007, P = 10.
#pragma once

#include <hip/hip_runtime.h>

namespace mdship {

template <typename T>
__device__ __forceinline__ void host_store(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void host_stores_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

}  // namespace mdship
