// Device-side work plan of the attention kernels over paged history (gfx950,
// wave64): which part of which request a workgroup takes.
//
// Request lengths live in device memory, so the host can only size a grid for
// the shapes.  One workgroup per (row, head) then takes as long as the
// longest request: a batch of 32 requests of 62..8000 tokens (a fifth of the
// tokens of 32 x 8192) took 113 us per residual-loop call against 161 us for
// the full batch; with the plan it takes 53 us, and the full batch, whose
// equal lengths stay unsplit, 161 us as before.  Every wave derives the same plan from the lengths: a chunk size
// that spreads the batch's total work over `target` workgroups per head, and
// ceil(length / chunk) near-equal splits per request.  The plan takes two
// DPP scans and no LDS or barrier (about 0.2 us once the lengths have
// arrived); workgroups past the planned items exit.
#pragma once

#include "rq_device.h"

namespace rq {

// Requests the plan covers (64 per register set); calls with more requests
// take the host's split count for every request.
constexpr int kPlanChunks = 4;
constexpr int kPlanRequests = 64 * kPlanChunks;

// One request's share: `count` items (rows, or row tiles) of `length` units
// each; `first` and `tokens` are carried to the item that is found.
struct PlanEntry {
    int count, length, first, tokens;
};

struct PlanItem {
    int request;  // -1: no work for this item
    int index;    // which of the request's `count` items
    int split, splits;
    int length, first, tokens;
    int offset;   // item index of split 0 of this (request, index)
    int total;    // items of the whole plan
};

template <int Ctrl>
__device__ __forceinline__ uint32_t plan_dpp(uint32_t x) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, Ctrl, 0xF, 0xF, true);
}

// Largest value of the wave, in every lane.
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
    x = max(x, plan_dpp<0xB1>(x));   // quad_perm [1,0,3,2]
    x = max(x, plan_dpp<0x4E>(x));   // quad_perm [2,3,0,1]
    x = max(x, plan_dpp<0x124>(x));  // row_ror:4
    x = max(x, plan_dpp<0x128>(x));  // row_ror:8
    return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, 16)),
               max(__builtin_amdgcn_readlane(x, 32), __builtin_amdgcn_readlane(x, 48)));
}

// Inclusive sum over lanes 0..lane of the wave.
__device__ __forceinline__ uint32_t wave_scan(uint32_t x, int lane) {
    x += plan_dpp<0x111>(x);  // row_shr:1, 2, 4, 8 (zero past the row)
    x += plan_dpp<0x112>(x);
    x += plan_dpp<0x114>(x);
    x += plan_dpp<0x118>(x);
    const uint32_t t0 = __builtin_amdgcn_readlane(x, 15), t1 = __builtin_amdgcn_readlane(x, 31),
                   t2 = __builtin_amdgcn_readlane(x, 47);
    return x + (lane >= 16 ? t0 : 0u) + (lane >= 32 ? t1 : 0u) + (lane >= 48 ? t2 : 0u);
}

// Item `item` of the plan over `requests` (at most kPlanRequests) requests.
// `entry(b)` returns request b's share (count 0 past the last request; its
// loads must be safe there).  chunk = max(min_chunk, ceil(total work /
// target)), at most max_chunk units per split (0 target: unsplit up to
// max_chunk); at most max_splits splits.  The items number at most target +
// the sum of the counts while max_chunk and max_splits do not bind (the host
// sizes the grid).  The host keeps the total work below 2^31.
// Wave-uniform; every wave of the grid computes the same plan.
template <class Entry>
__device__ __forceinline__ PlanItem plan_item(int requests, int item, int target, int min_chunk, int max_chunk,
                                              int max_splits, Entry entry) {
    const int lane = threadIdx.x & 63;
    PlanEntry e[kPlanChunks];
    uint32_t work = 0, longest = 0;
    bool single = true;
#pragma unroll
    for (int j = 0; j < kPlanChunks; ++j) {
        e[j] = PlanEntry{0, 0, 0, 0};
        if (64 * j < requests) e[j] = entry(64 * j + lane);
        work += (uint32_t)e[j].count * (uint32_t)e[j].length;
        longest = max(longest, (uint32_t)e[j].length);
        single = single && e[j].count == (64 * j + lane < requests ? 1 : 0);
    }
    const uint32_t total = __builtin_amdgcn_readlane(wave_scan(work, lane), 63);
    longest = wave_max_u32(longest);
    uint32_t chunk = (uint32_t)max_chunk;
    // Plain batches whose longest request is at most a chunk (equal lengths
    // that fill the device): item i is request i, and no division is taken.
    if (requests <= 64 && longest <= (uint32_t)max_chunk && __all(single) &&
        (target <= 0 || longest <= (uint32_t)min_chunk ||
         (uint64_t)(longest - 1) * (uint32_t)target < total)) {
        PlanItem r{item < requests ? item : -1, 0, 0, 1, 0, 0, 0, item, requests};
        const int src = item < requests ? item : 0;
        r.length = __builtin_amdgcn_readlane(e[0].length, src);
        r.first = __builtin_amdgcn_readlane(e[0].first, src);
        r.tokens = __builtin_amdgcn_readlane(e[0].tokens, src);
        return r;
    }
    if (target > 0) {
        const uint32_t even = (total + (uint32_t)target - 1) / (uint32_t)target;
        chunk = even > (uint32_t)min_chunk ? even : (uint32_t)min_chunk;
        chunk = chunk < (uint32_t)max_chunk ? chunk : (uint32_t)max_chunk;
    }
    PlanItem r{-1, 0, 0, 1, 0, 0, 0, 0, 0};
    uint32_t base = 0;
#pragma unroll
    for (int j = 0; j < kPlanChunks; ++j) {
        if (64 * j >= requests) break;
        uint32_t splits = ((uint32_t)e[j].length + chunk - 1) / chunk;
        splits = splits < 1u ? 1u : splits;
        splits = splits < (uint32_t)max_splits ? splits : (uint32_t)max_splits;
        const uint32_t items = (uint32_t)e[j].count * splits;
        const uint32_t end = base + wave_scan(items, lane), begin = end - items;
        const uint64_t mask = __ballot(begin <= (uint32_t)item && (uint32_t)item < end);
        if (mask != 0) {
            const int src = __builtin_ctzll(mask);
            r.request = 64 * j + src;
            r.splits = (int)__builtin_amdgcn_readlane(splits, src);
            const uint32_t local = (uint32_t)item - __builtin_amdgcn_readlane(begin, src);
            r.index = (int)(local / (uint32_t)r.splits);
            r.split = (int)local - r.index * r.splits;
            r.offset = item - r.split;
            r.length = __builtin_amdgcn_readlane(e[j].length, src);
            r.first = __builtin_amdgcn_readlane(e[j].first, src);
            r.tokens = __builtin_amdgcn_readlane(e[j].tokens, src);
        }
        base = __builtin_amdgcn_readlane(end, 63);
    }
    r.total = (int)base;
    return r;
}

// The first unit of split `split` of `splits` near-equal parts of `length` units.
__device__ __forceinline__ int split_begin(int length, int split, int splits) {
    const int each = length / splits, rest = length - each * splits;
    return split * each + (split < rest ? split : rest);
}

// ------------------------------------------------------------------ arrivals
//
// The workgroup that finishes last of a split item merges, so the splits of
// an item count themselves in one 64-bit word of the call's workspace: the
// upper 56 bits hold the call's tag, the lower 8 the arrivals so far.  Every
// split first makes sure that the word carries the tag (tag_arrivals, early
// in its prologue: a word whose tag is not this call's is replaced by an
// empty one), so the word needs no clearing launch before the call (5 us with
// its gap) and the arrival itself is one atomic add.  The last arrival writes
// 0, so a replay of a captured call, which repeats the tag, starts from an
// untagged word as well.  Tags come from a process-wide counter with a random
// start (next_call_tag in capi.hip): stale memory equals a call's tag with
// probability 2^-56.

// The word as an early load of thread 0 saw it (issued where its latency is hidden).
__device__ __forceinline__ uint64_t peek_arrivals(const uint64_t* word) {
    return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Thread 0 of every split, before its arrival: the word carries `tag` afterwards.
// A failed exchange means that the word has changed since `seen`, which only
// another split of this call does, and only to a tagged word.
__device__ __forceinline__ void tag_arrivals(uint64_t* word, uint64_t tag, uint64_t seen) {
    if ((seen >> 8) != tag)
        (void)__hip_atomic_compare_exchange_strong(word, &seen, tag << 8, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
}

// Counts this workgroup (after every thread's handoff stores) and returns
// true in every thread of the workgroup that arrives last of `expected`.
// Nothing waits for other workgroups.
__device__ __forceinline__ bool arrive_last_tagged(uint64_t* word, int expected, int* lds_flag) {
    wait_vector_memory();
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint64_t before = __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = (int)(before & 0xff) == expected - 1;
        if (last) __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *lds_flag = last;
    }
    __syncthreads();
    return *lds_flag != 0;
}

}  // namespace rq
