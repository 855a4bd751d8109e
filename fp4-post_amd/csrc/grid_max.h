// A maximum over all workgroups of one launch (single-launch quantizer, nvfp4_quant.hip; resident round trip, nvfp4_roundtrip.hip).
#pragma once
#include "metis_device.h"
#include "metis_host.h"

namespace metis {

// ---------------------------------------------------------------------------------------------
// The grid-wide maximum does not assume that all workgroups are resident together.  Workgroups arrive through a
// two-level tree (64 groups of up to 64 workgroups) whose nodes are a maximum and an arrival counter, each updated by one
// read-modify-write, so exactly one workgroup learns that it is the LAST to arrive and what the tensor maximum is.  It
// exchanges {call tag, result, maximum} into 64 words (one per group, a line each) and cleans the tree for the next call.  Every other workgroup polls its group's word a bounded number of times.  One that gives
// up -- because part of the grid is still waiting for a compute unit, held by another kernel or by these very pollers
// -- raises its flag, swaps {call tag, "somebody left"} into its group's word and exits WITHOUT the output that waits for
// the maximum: the last workgroup finds that marker in what its exchange returns and writes that output itself.  If the
// exchange came first, the leaver's swap fails, it reads the result and finishes after all.  That decision hangs on one word, so relaxed device-scope atomics suffice on the ordinary path (an
// acquire or release at device scope writes back or invalidates a whole L2 on this part); only a workgroup that leaves
// and the last workgroup that cleans up after one pay for fences.  Every wave exits after a bounded time whatever else
// runs on the device, and the result is always complete and always the same bytes as the two-launch path.
// The area starts zero-filled; a call leaves the tree clean and only tagged words behind.
// What giving up costs: the polls (up to a few milliseconds), then one workgroup writes for all that left, at the speed of one.  The round
// trip keeps its grid to half of the device, where this was not seen beside any other work; the single-launch quantizer is for callers
// that have the device to themselves.
// ---------------------------------------------------------------------------------------------
constexpr uint32_t kSpinLimit = 4096;            // polls (roughly a microsecond each) before a workgroup leaves its output behind
constexpr uint32_t kGroups = 64;                 // groups, and the most members a group can have
constexpr int kFusedMaxGrid = kGroups * kGroups;
// locations inside the synchronisation area (uint32 units)
__device__ __forceinline__ uint64_t* sync_generation(uint32_t* s) { return reinterpret_cast<uint64_t*>(s); }
__device__ __forceinline__ uint32_t* sync_top(uint32_t* s) { return s + 4; }                           // {maximum, arrivals}
__device__ __forceinline__ uint32_t* sync_group(uint32_t* s, uint32_t j) { return s + 64 + j * 32; }     // {maximum, arrivals}, a line each
__device__ __forceinline__ uint64_t* sync_result(uint32_t* s, uint32_t j) { return reinterpret_cast<uint64_t*>(s + 2176 + j * 32); }
__device__ __forceinline__ uint32_t* sync_left_flag(uint32_t* s, uint32_t b) { return s + 4224 + b; }
static_assert((4224 + kFusedMaxGrid) * 4 <= kWsSyncBytes, "synchronisation area too small");

#define METIS_AT_LOAD(p) __hip_atomic_load((p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define METIS_AT_STORE(p, v) __hip_atomic_store((p), (v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define METIS_AT_CAS(p, expected, desired) \
    __hip_atomic_compare_exchange_strong((p), (expected), (desired), __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
#define METIS_AT_XCHG(p, v) __hip_atomic_exchange((p), (v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)

// a group's result word: tag << 18 | kind << 16 | bf16 payload; kind 0: the tensor maximum, kind 1: a member has left
__device__ __forceinline__ uint64_t result_word(uint64_t tag, uint32_t kind, uint32_t payload) { return (tag << 18) | ((uint64_t)kind << 16) | payload; }
__device__ __forceinline__ bool is_result(uint64_t w, uint64_t tag) { return (w >> 16) == (tag << 2); }
__device__ __forceinline__ bool is_left_marker(uint64_t w, uint64_t tag) { return (w >> 16) == ((tag << 2) | 1u); }

// The same for maxima that need not be bf16 values, in words of their own (a word of one form can look like a later call's word of the
// other): tag << 33 | kind << 32 | binary32 payload.
__device__ __forceinline__ uint64_t* sync_result32(uint32_t* s, uint32_t j) { return reinterpret_cast<uint64_t*>(s + 4224 + kFusedMaxGrid + j * 32); }
static_assert((4224 + kFusedMaxGrid + kGroups * 32) * 4 <= kWsSyncBytes, "synchronisation area too small");
template <bool F32> struct ResultWord {
    static __device__ __forceinline__ uint64_t* slot(uint32_t* s, uint32_t j) { return F32 ? sync_result32(s, j) : sync_result(s, j); }
    static __device__ __forceinline__ uint64_t result(uint64_t tag, float m)
    {
        return F32 ? (tag << 33) | __float_as_uint(m) : result_word(tag, 0u, __float_as_uint(m) >> 16);
    }
    static __device__ __forceinline__ uint64_t marker(uint64_t tag) { return F32 ? (tag << 33) | ((uint64_t)1u << 32) : result_word(tag, 1u, 0u); }
    static __device__ __forceinline__ bool has_result(uint64_t w, uint64_t tag) { return F32 ? (w >> 32) == (tag << 33) >> 32 : is_result(w, tag); }
    static __device__ __forceinline__ bool has_marker(uint64_t w, uint64_t tag) { return F32 ? (w >> 32) == marker(tag) >> 32 : is_left_marker(w, tag); }
    static __device__ __forceinline__ float value(uint64_t w) { return __uint_as_float(F32 ? (uint32_t)w : ((uint32_t)w & 0xffffu) << 16); }
};

struct GridMaxState {
    float wave_part[4];
    uint32_t last;               // this workgroup was the last to arrive
    uint32_t known;              // result holds the tensor maximum
    float result;
    uint32_t nleft;
    uint32_t left[256];          // workgroups of one slab of 256 flags that left their output behind
};

// Every thread, at kernel start (before its workgroup arrives, so before the counter can move): the tag of this call.
__device__ __forceinline__ uint64_t grid_max_begin(uint32_t* sync)
{
    return METIS_AT_LOAD(sync_generation(sync)) + 1u;
}

// One more arrival with maximum `bits` at a tree node {maximum, arrivals}; true for the arrival that completes `expected`,
// with the node's maximum.  Two relaxed read-modify-writes without retry: the counter's increment is made to depend on
// the value the maximum's returns, so it is issued only after the maximum has been performed at the coherence point; the
// arrival that sees the count complete therefore reads a maximum that every earlier arrival has folded in.
__device__ __forceinline__ bool tree_arrive(uint32_t* node, uint32_t bits, uint32_t expected, uint32_t& folded)
{
    const uint32_t before = __hip_atomic_fetch_max(node, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t one = 1u + (before >> 31);                      // bit 31 of a non-negative float's pattern: always 0
    if (__hip_atomic_fetch_add(node + 1, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != expected - 1u) return false;
    folded = METIS_AT_LOAD(node);
    METIS_AT_STORE(node, 0u);                                      // nobody else touches the node before the next call
    METIS_AT_STORE(node + 1, 0u);
    return true;
}

// Called by every thread of every workgroup, once: folds the workgroup maximum (a bf16 or binary32 value, not negative) into the tree.
__device__ __forceinline__ void grid_max_arrive(float thread_max, uint32_t* sync, GridMaxState& sh)
{
    const float m = wave_max(thread_max);
    if ((threadIdx.x & 63) == 0) sh.wave_part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t bits = __float_as_uint(fmaxf(fmaxf(sh.wave_part[0], sh.wave_part[1]), fmaxf(sh.wave_part[2], sh.wave_part[3])));
        const uint32_t j = blockIdx.x % kGroups;
        const uint32_t ngroups = gridDim.x < kGroups ? gridDim.x : kGroups;
        const uint32_t members = (gridDim.x + kGroups - 1u - j) / kGroups;
        uint32_t gm = 0u, fin = 0u;
        const bool last = tree_arrive(sync_group(sync, j), bits, members, gm) && tree_arrive(sync_top(sync), gm, ngroups, fin);
        sh.last = last ? 1u : 0u;
        sh.known = sh.last;
        sh.result = __uint_as_float(fin);
    }
}

}  // namespace metis
