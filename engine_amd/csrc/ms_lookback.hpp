// ms_lookback.hpp -- prefix sums over the tiles of one launch.
//
// A kernel whose output offsets depend on every tile before it takes its
// tiles in ticket order and publishes one 64-bit word per tile: first the
// tile's own total, then (once known) the total of all tiles up to it.  A
// tile's offset is found by one wave reading 64 predecessors' words at a
// time.  Progress: tickets are handed out in order to workgroups that already
// run.  A kernel that looks back for the tile it holds (k_merge, k_rle_starts)
// publishes that tile's total first.  One that looks back a tile late
// (k_emit_onepass, k_rle_onepass, k_select_onepass) holds up to three tickets:
// the tile that waits for its offset, a later one whose total it publishes
// before that wait, and the next one, whose total comes after it.  In both a
// workgroup only ever waits for words of tiles below one that it has published
// itself, and its tickets ascend; so the owner of the lowest unpublished tile
// waits, if at all, for published words only, and goes on to publish.  Totals
// are enough for that: a wait ends with the words of all tiles below, prefix
// or not.  The page starts of k_emit_onepass are words of the same kind, stored
// by a page's first tile at its own look-back and waited for by the page's
// later tiles after theirs: the lowest tile whose look-back is not done waits
// for no page start that is not stored.
// The words and the ticket counter are cleared before the launch.
#pragma once

#include "ms_device.hpp"

namespace ms {

constexpr uint64_t LB_TOTAL = 1ull << 62;      // the tile's own total
constexpr uint64_t LB_PREFIX = 2ull << 62;     // the total up to and with the tile
constexpr uint64_t LB_VALUE = LB_TOTAL - 1ull;

__device__ __forceinline__ uint64_t lb_load(const uint64_t *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void lb_store(uint64_t *p, uint64_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The next ticket of a launch (one thread).
__device__ __forceinline__ uint64_t lb_ticket(uint64_t *counter)
{
    return __hip_atomic_fetch_add(counter, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Publishes a tile's own total (below 2^62; one wave).
__device__ __forceinline__ void lb_publish(uint64_t *words, uint64_t tile, uint64_t total)
{
    if (lane_id() == 0) lb_store(words + tile, (tile ? LB_TOTAL : LB_PREFIX) | total);
}

// Sum of the totals of tiles 0 .. tile - 1, after lb_publish of this tile's
// `total`, in two halves (all 64 lanes of one wave): lb_request asks for
// the words of the 64 LB_SPAN tiles in front, lb_exclusive waits for them.
// Loads return in order, so what a wave loads between the two does not
// delay its words; a step past them does wait for it.
constexpr uint32_t LB_SPAN = 2;

__device__ __forceinline__ void lb_request(const uint64_t *words, int64_t last, uint64_t (&w)[LB_SPAN])
{
#pragma unroll
    for (uint32_t i = 0; i < LB_SPAN; i++) {
        const int64_t k = last - (int64_t)(64 * i + lane_id());
        w[i] = k >= 0 ? lb_load(words + k) : LB_PREFIX;
    }
}

__device__ __forceinline__ uint64_t lb_exclusive(uint64_t *words, uint64_t tile, uint64_t total,
                                                 uint64_t (&w)[LB_SPAN])
{
    const uint32_t t = lane_id();
    if (tile == 0) return 0;
    uint64_t sum = 0;
    for (int64_t last = (int64_t)tile - 1;;) {   // the nearest word of the step: row 0, lane 0
        bool found = false;
#pragma unroll
        for (uint32_t i = 0; i < LB_SPAN; i++) {
            if (found) continue;
            // wait for the row's words up to its nearest prefix
            uint64_t pre;
            for (;;) {
                pre = __ballot((w[i] & LB_PREFIX) != 0);
                const uint64_t none = __ballot(w[i] == 0);
                if ((none & (pre ? (pre & (0ull - pre)) - 1ull : ~0ull)) == 0) break;
                __builtin_amdgcn_s_sleep(1);
                if (w[i] == 0) w[i] = lb_load(words + (last - (int64_t)(64 * i + t)));
            }
            const uint32_t stop = pre ? (uint32_t)__builtin_ctzll(pre) : 63u;
            sum += t <= stop ? w[i] & LB_VALUE : 0ull;
            found = pre != 0;
        }
        if (found) break;
        last -= 64 * LB_SPAN;
        lb_request(words, last, w);
    }
    sum = wave_sum_u64(sum);
    if (t == 0) lb_store(words + tile, LB_PREFIX | (sum + total));
    return sum;
}

}  // namespace ms
