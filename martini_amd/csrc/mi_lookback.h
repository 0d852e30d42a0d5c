// Running totals over work groups in one pass, by decoupled look-back (Merrill and
// Garland, "Single-pass Parallel Prefix Scan with Decoupled Look-back", 2016).
//
// Work groups are numbered by a ticket, publish their own count in a 64-bit word
// (state and value together, so no other memory needs ordering) and sum the words
// before theirs, back to the nearest one that holds a total.  A group waits only for
// lower tickets, which run already and publish before they wait.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mi {

// Look-back words: state in the top bits, a count in the rest (of the group
// alone, or of all groups up to it).
constexpr unsigned long long LB_GROUP = 1ull << 62, LB_ALL = 2ull << 62;
constexpr unsigned long long LB_STATE = 3ull << 62;

// Pause between two looks at words that are not published yet (x 64 cycles):
// the groups that wait would otherwise fill the fabric with their reads.
constexpr int LOOK_SLEEP = 8;

__device__ inline unsigned long long look_load(const unsigned long long* w) {
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void look_store(unsigned long long* w, unsigned long long v) {
    __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sum of the counts of the groups before `group`, taken by one wave, 64 words
// at a time.
__device__ inline unsigned long long look_back(const unsigned long long* look, int64_t group) {
    const int lane = threadIdx.x & 63;
    unsigned long long base = 0;
    for (int64_t j = group - 1; j >= 0; j -= 64) {
        unsigned long long v;
        uint64_t all, need;
        while (true) {
            v = j - lane >= 0 ? look_load(&look[j - lane]) : LB_ALL;
            all = __ballot((v & LB_STATE) == LB_ALL);
            need = all ? (all & (0ull - all)) * 2ull - 1ull : ~0ull;  // up to the nearest total
            if ((__ballot((v & LB_STATE) != 0ull) & need) == need) break;
            __builtin_amdgcn_s_sleep(LOOK_SLEEP);
        }
        unsigned long long x = (need >> lane) & 1ull ? v & ~LB_STATE : 0ull;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) x += __shfl_xor(x, d, 64);
        base += x;
        if (all) break;
    }
    return base;
}

}  // namespace mi
