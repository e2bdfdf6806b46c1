// The last workgroup of a launch, found without a fence and without one counter for all.
//
// Workgroups publish what the last one combines by device-scope atomics whose results they wait for, so
// that nothing has to be written back (a device-scope fence per workgroup writes back the L2 cache with
// all that the workgroup stored: 20.6 against 13.0 us for a 129 x 65 x 33 refinement step of 510
// workgroups).  Atomics on one address follow each other at about 5 ns: they count themselves in in
// kGridGroups groups first, each with a cache line of its own (a Jacobi sweep of 510
// workgroups with two atomics each: 21.6 -> 18.0 us).
#pragma once

#include <hip/hip_runtime.h>

namespace sr {

constexpr int kGridGroups = 16;
constexpr int kGridWords = 32 * (kGridGroups + 1);   // unsigned words, 0 before the first launch

__device__ inline unsigned grid_group() { return blockIdx.x % kGridGroups; }

// result of an atomic on which the next one has to wait
template <typename T>
__device__ __forceinline__ void arrived(T v) {
    asm volatile("" : : "v"(v) : "memory");
}

// By one thread of each workgroup: whether all others have been here.  words are 0 again afterwards.
__device__ inline bool grid_last(unsigned *words) {
    const unsigned g = grid_group(), in_group = (gridDim.x - g + kGridGroups - 1) / kGridGroups;
    unsigned *const w = words + 32 * (1 + g);
    if (__hip_atomic_fetch_add(w, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != in_group - 1) return false;
    __hip_atomic_store(w, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned groups = min(gridDim.x, (unsigned)kGridGroups);
    if (__hip_atomic_fetch_add(words, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != groups - 1) return false;
    __hip_atomic_store(words, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

}  // namespace sr
