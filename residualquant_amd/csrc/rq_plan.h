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
// ceil(length / chunk) near-equal splits per request.  The plan takes a few
// DPP scans and no LDS or barrier (about 0.2 us for near-equal requests, 0.7
// us else, once the lengths have arrived); workgroups past the planned items
// exit.
#pragma once

#include "rq_device.h"
#include "rq_kernels.h"

namespace rq {

// Requests the plan covers, one per lane; calls with more requests take the
// host's split count for every request.
constexpr int kPlanRequests = 64;

// One request's share: `count` items (rows, or row tiles) of `length` units
// each, `rows` rows in all; `first` and `tokens` are carried to the item that
// is found.
struct PlanEntry {
    int count, length, first, tokens, rows;
};

struct PlanItem {
    int request;  // -1: no work for this item
    int index;    // which of the request's `count` items
    int split, splits;
    int length, first, tokens, rows;
    int offset;   // item index of split 0 of this (request, index)
    int entry;    // rows x splits of the requests before this one
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

// The sizes of a plan.  A batch whose longest request is at most 9/8 of the
// mean takes `even_splits` of every request, the count the host chose for
// equal lengths as long as the page table, or fewer so that a split keeps
// min_chunk units.  Else a request takes ceil(length / chunk) splits (at most
// max_splits), chunk = max(min_chunk, ceil(total work / target)) units, at
// most max_chunk (target 0: max_chunk), and at least round_chunk where smaller
// ones would make more items than round_target; the items are ordered by size
// in four classes, the longest first, so that what starts last is short.
// A batch whose counts already are 3/4 of the target counts as near equal up
// to full_eighths / 8 of the mean: 13 for several rows per request (6 requests
// of 1310..4150 tokens x 29 rows x 55 heads: 94 us with the two even splits,
// 100 us with nine planned ones), 18 for decode (42 requests of 188..922
// tokens, 16 heads: 4-loop step 114 us whole, 125 us planned; 64 requests of
// 100..2000 tokens, the longest 3.2 times the mean: residual call 62 us whole,
// 54 us planned).
struct PlanSizes {
    int target, even_splits, min_chunk, max_chunk, max_splits;
    int round_chunk, round_target;
    int full_eighths;
    int whole_length;  // near-equal requests of at most this many units stay whole
};

// What every request of a plan shares.
struct PlanShare {
    bool even, whole;  // near-equal requests; of one split each
    uint32_t even_splits, chunk;
};

// `total`: count x length over the requests, `counts` their counts, `longest`
// the longest length with a count.
__host__ __device__ __forceinline__ PlanShare plan_share_of(const PlanSizes& sizes, uint32_t total, uint32_t counts,
                                                            uint32_t longest) {
    const uint32_t min_chunk = (uint32_t)sizes.min_chunk;
    PlanShare s;
    const bool full = 4ull * counts >= 3ull * (uint32_t)sizes.target;
    s.even = 8ull * longest * counts <= (uint64_t)(full ? sizes.full_eighths : 9) * total;
    s.even_splits = (uint32_t)sizes.even_splits;
    if (s.even_splits > 1 && longest < s.even_splits * min_chunk) s.even_splits = max(longest / min_chunk, 1u);
    if (sizes.whole_length > 0 && longest <= (uint32_t)min(sizes.whole_length, sizes.max_chunk)) s.even_splits = 1;
    s.chunk = (uint32_t)sizes.max_chunk;
    if (s.even && s.even_splits == 1 && 8ull * longest * counts > 9ull * total && longest <= s.chunk) {
        // Whole, but not alike: one split each, the longest first.
        s.even = s.whole = false;
        s.chunk = longest;
        return s;
    }
    s.whole = s.even && s.even_splits == 1;
    if (!s.even && sizes.target > 0) {
        const uint32_t share = (total + (uint32_t)sizes.target - 1) / (uint32_t)sizes.target;
        const uint32_t round_share = (total + (uint32_t)sizes.round_target - 1) / (uint32_t)sizes.round_target;
        s.chunk = min(max(max(share, min_chunk), min((uint32_t)sizes.round_chunk, round_share)), s.chunk);
    }
    return s;
}

__device__ __forceinline__ PlanShare plan_share(const PlanSizes& sizes, const PlanEntry& own, int lane) {
    const uint32_t length = (uint32_t)own.length, count = (uint32_t)own.count;
    return plan_share_of(sizes, __builtin_amdgcn_readlane(wave_scan(count * length, lane), 63),
                         __builtin_amdgcn_readlane(wave_scan(count, lane), 63), wave_max_u32(count > 0 ? length : 0u));
}

__host__ __device__ __forceinline__ uint32_t plan_splits(const PlanSizes& sizes, const PlanShare& share, uint32_t length) {
    if (share.even) return share.even_splits;
    uint32_t splits = min(max((length + share.chunk - 1) / share.chunk, 1u), (uint32_t)sizes.max_splits);
    if (splits > 1 && splits * (uint32_t)sizes.min_chunk > length && length <= (uint32_t)sizes.max_chunk) splits -= 1;
    return splits;
}

// Item `key` of the plan over `requests` (at most kPlanRequests) requests.
// `own` is the share of request `lane` (count 0 past the last request).  The items number at
// most max(even_splits x counts, target + counts) while max_chunk does not
// bind (the host sizes the grid), and the entries (rows x splits) at most
// max(even_splits x rows, rows + target x the most rows of one item).  The
// host keeps the total work below 2^31.  Wave-uniform; every wave of every
// kernel of a call derives the same plan.
__device__ __forceinline__ PlanItem plan_find(int requests, int key, const PlanSizes& sizes, const PlanEntry& own) {
    const int lane = threadIdx.x & 63;
    const uint32_t length = (uint32_t)own.length, count = (uint32_t)own.count;
    const PlanShare share = plan_share(sizes, own, lane);
    PlanItem r{-1, 0, 0, 1, 0, 0, 0, 0, 0, 0, 0};
    auto take = [&](int src) {
        r.request = src;
        r.length = __builtin_amdgcn_readlane(own.length, src);
        r.first = __builtin_amdgcn_readlane(own.first, src);
        r.tokens = __builtin_amdgcn_readlane(own.tokens, src);
        r.rows = __builtin_amdgcn_readlane(own.rows, src);
    };
    // Plain batches of near-equal requests that stay whole: item i is request i.
    if (share.whole && __all(own.count == (lane < requests ? 1 : 0))) {
        if (key < requests) take(key);
        r.entry = (int)(__builtin_amdgcn_readlane(wave_scan((uint32_t)own.rows, lane), key & 63)) - r.rows;
        r.offset = key;
        r.total = requests;
        return r;
    }
    const uint32_t splits = plan_splits(sizes, share, length);
    int size_class = 0;
    if (!share.even) {
        // A split's share of a chunk: above 3/4, 1/2, 1/4 or less.
        const float whole = (float)splits * (float)share.chunk, part = (float)length;
        size_class = part > 0.75f * whole ? 0 : part > 0.5f * whole ? 1 : part > 0.25f * whole ? 2 : 3;
    }
    const uint32_t entry_end = wave_scan((uint32_t)own.rows * splits, lane);
    uint32_t local = 0, base = 0;
    for (int k = 0; k < (share.even ? 1 : 4); ++k) {
        const uint32_t items = size_class == k ? count * splits : 0u;
        const uint32_t end = base + wave_scan(items, lane), begin = end - items;
        const uint64_t mask = __ballot(begin <= (uint32_t)key && (uint32_t)key < end);
        if (mask != 0) {
            take(__builtin_ctzll(mask));
            r.offset = (int)__builtin_amdgcn_readlane(begin, r.request);
            local = (uint32_t)(key - r.offset);
        }
        base = __builtin_amdgcn_readlane(end, 63);
    }
    r.total = (int)base;
    if (r.request < 0) return r;
    r.splits = (int)__builtin_amdgcn_readlane(splits, r.request);
    r.index = (int)(local / (uint32_t)r.splits);
    r.split = (int)local - r.index * r.splits;
    r.offset += r.index * r.splits;
    r.entry = (int)__builtin_amdgcn_readlane(entry_end, r.request) - r.rows * r.splits;
    return r;
}

// The splits and the first entry of request `request` in the same plan.
struct PlanRequest {
    int splits, entry;
};

__device__ __forceinline__ PlanRequest plan_request(int request, const PlanSizes& sizes, const PlanEntry& own) {
    const int lane = threadIdx.x & 63;
    const PlanShare share = plan_share(sizes, own, lane);
    const uint32_t splits = share.whole ? 1u : plan_splits(sizes, share, (uint32_t)own.length);
    const uint32_t entry_end = wave_scan((uint32_t)own.rows * splits, lane);
    PlanRequest r;
    r.splits = (int)__builtin_amdgcn_readlane(splits, request);
    r.entry = (int)__builtin_amdgcn_readlane(entry_end, request) - __builtin_amdgcn_readlane(own.rows, request) * r.splits;
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
// upper 48 bits hold the call's tag, the lower 16 the arrivals so far (a long
// page table makes several hundred splits of a request's several rows: the
// host takes at most kMaxArrivals).  Every split first makes sure that the word carries the tag (tag_arrivals, early
// in its prologue: a word whose tag is not this call's is replaced by an
// empty one), so the word needs no clearing launch before the call (5 us with
// its gap) and the arrival itself is one atomic add.  The last arrival writes
// 0, so a replay of a captured call, which repeats the tag, starts from an
// untagged word as well.  Tags come from a process-wide counter with a random
// start (next_call_tag in capi.hip): stale memory equals a call's tag with
// probability 2^-48.

// The word as an early load of thread 0 saw it (issued where its latency is hidden).
__device__ __forceinline__ uint64_t peek_arrivals(const uint64_t* word) {
    return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Thread 0 of every split, before its arrival: the word carries `tag` afterwards.
// A failed exchange means that the word has changed since `seen`, which only
// another split of this call does, and only to a tagged word.
__device__ __forceinline__ void tag_arrivals(uint64_t* word, uint64_t tag, uint64_t seen) {
    if ((seen >> kArrivalBits) != tag)
        (void)__hip_atomic_compare_exchange_strong(word, &seen, tag << kArrivalBits, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
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
        const bool last = (int)(before & kMaxArrivals) == expected - 1;
        if (last) __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *lds_flag = last;
    }
    __syncthreads();
    return *lds_flag != 0;
}

}  // namespace rq
