// The workgroups that share a sum over K (or over keys) leave their parts in a workspace, and the last one to arrive adds them up
// in order: one launch instead of two, whose second one costs 3 to 5 us.  Nobody waits for anybody.
//
// The count of arrivals lives in the caller's workspace, whose contents are unknown and which other tensors may have used in
// between.  Each launch therefore brings a tag, 56 bits that no other launch of the process has: a workgroup that finds
// another tag in the word replaces it by its own with a count of zero (compare-and-swap, at its start, while its operands are on
// their way), the last one clears the word.  A captured launch keeps its tag, which the cleared word allows: every replay starts
// from a word without it.
//
// Parts and counts go past the L2s of the XCDs, which are not coherent with one another inside a launch: stores and loads at agent
// scope (the sc1 bit), each wave waiting for its own stores in front of the barrier that the arrival is counted behind.
#pragma once
#include "gemm_common.h"

namespace mhip {

// A tag for a launch: never zero, the low eight bits clear (runtime.hip).
uint64_t launch_tag();

constexpr int kAgentScope = 16;            // sc1 of a buffer access

__device__ __forceinline__ __amdgpu_buffer_rsrc_t parts_rsrc(const void* p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, 0x7FFFFFFF, 0x00020000);
}
__device__ __forceinline__ void store_part(__amdgpu_buffer_rsrc_t r, uint32_t byte, f32x4 v) {
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, byte, 0, kAgentScope);
}
__device__ __forceinline__ f32x4 load_part(__amdgpu_buffer_rsrc_t r, uint32_t byte) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, byte, 0, kAgentScope));
}

__device__ __forceinline__ void store_part(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float load_part(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// By one thread: the word as it is at the workgroup's start (asked for before its operands are), and, once that is there, the claim.
__device__ __forceinline__ uint64_t arrive_look(const uint64_t* word) {
    return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void arrive_claim(uint64_t* word, uint64_t seen, uint64_t tag) {
    // (a swap that fails has met the tag: only workgroups of this launch write the word)
    if ((seen & ~(uint64_t)255) != tag)
        __hip_atomic_compare_exchange_strong(word, &seen, tag, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// By the whole workgroup, when its word is claimed and its part is stored: whether all `parts` workgroups (255 at most) have come by now.  `flag`: a word of LDS.
__device__ __forceinline__ bool arrive_last(uint64_t* word, int parts, int* flag) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint64_t before = __hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = (int)(before & 255) == parts - 1;
        if (last) __hip_atomic_store(word, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last;
    }
    __syncthreads();
    asm volatile("" ::: "memory");
    return *flag != 0;
}

}  // namespace mhip
