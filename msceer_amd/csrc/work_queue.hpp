// Work queue of the re-integration pass (pass 3 of integrate.hip).
//
// q.busy counts the waves that hold work and the traces ahead whose vertex has
// been reached meanwhile ("wanted"), so that a wave left with nothing but
// traces ahead knows when nothing can want them any more.  The order of the
// steps makes a zero mean that:
//   a wave is counted before it claims anything (queue_enter, queue_claim) and
//   until it holds nothing and all it queued is in q.tail;
//   a trace ahead is counted by the wave that wants it, while that wave is
//   counted itself, until the wave that traced it has taken it over
//   (queue_takeover) and is counted in its place;
//   queue_drained reads the head, then the count, then the tail again: where
//   all slots reserved were claimed, none was reserved since and the count is
//   zero in between, no wave held work at that moment, and only one that does
//   can queue more.
#pragma once
#include <stdint.h>

namespace msceer {

// Re-integration work queue: `items` (capacity entries, 0xFFFFFFFF until
// written) and its claim/reserve counters.
struct WorkQueue {
    uint32_t* items;
    uint32_t capacity;
    uint32_t* head;         // next slot of the items queued during pass 3
    uint32_t* tail;         // slots reserved
    uint32_t* overflow;
    uint32_t* ahead_on;     // set once pass 3 traces vertices ahead
    uint32_t* chunk_head;   // next chunk of the items pass 2 queued
    uint32_t* first_count;  // items pass 2 queued
    uint32_t* busy;         // waves that hold anything but traces ahead, and traces ahead that are wanted
};

__device__ __forceinline__ uint32_t load_agent(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The functions below are one lane's, for its wave.

// Counts the wave; what it claims after that is claimed later in memory too.
__device__ __forceinline__ void queue_enter(const WorkQueue& q) {
    atomicAdd(q.busy, 1u);
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#endif
}

// Claims up to `want` of the reserved slots, from *base on; returns how many
// (none, too, where another wave was first).  The wave is then counted.
__device__ __forceinline__ uint32_t queue_claim(const WorkQueue& q, uint32_t want, bool& counted, uint32_t* base) {
    uint32_t h = load_agent(q.head);
    uint32_t t = load_agent(q.tail);
    t = t < q.capacity ? t : q.capacity;
    if (h >= t) return 0;
    if (!counted) queue_enter(q);
    counted = true;
    const uint32_t k = t - h < want ? t - h : want;
    if (!__hip_atomic_compare_exchange_strong(q.head, &h, h + k, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                              __HIP_MEMORY_SCOPE_AGENT))
        return 0;
    *base = h;
    return k;
}

// n traces ahead that are wanted become the wave's own work.
__device__ __forceinline__ void queue_takeover(const WorkQueue& q, uint32_t n, bool& counted) {
    if (!counted) n--;  // one count becomes the wave's
    counted = true;
    if (n) atomicAdd(q.busy, 0u - n);
}

// No wave holds work, no trace ahead is wanted and no slot is left.
__device__ __forceinline__ bool queue_drained(const WorkQueue& q) {
    const uint32_t t = load_agent(q.tail);
    if (load_agent(q.head) < (t < q.capacity ? t : q.capacity)) return false;
    if (load_agent(q.busy) != 0u) return false;
    return load_agent(q.tail) == t;
}

}  // namespace msceer
