// ms_merge_path.hpp -- how merge_sorted's tiles are cut: the split of the
// merged order between two lists and a tile's part of each.  Index
// arithmetic only, so that it can be checked on the host.
#pragma once

#include <stdint.h>

namespace ms {

// The i-th of 64 places probed in [lo, lo + span).
__host__ __device__ __forceinline__ uint64_t merge_probe(uint64_t lo, uint64_t span, uint32_t i)
{
    return span <= 64 ? lo + i : lo + span * i / 64;
}

// Values of a (na of them) among the first d of the merged order of a and
// b (nb).  count(lo, span, d) = how many of the 64 probes k of [lo, lo + span)
// lie in it and have a[k] <= b[d - 1 - k]; with ascending lists those are the
// first ones.  Whatever count says, the result lies in
// [max(d, nb) - nb, min(d, na)], so that d minus it is a place of b.
template <class Count>
__host__ __device__ __forceinline__ uint64_t merge_split(uint64_t na, uint64_t nb, uint64_t d, const Count &count)
{
    uint64_t lo = d > nb ? d - nb : 0, hi = d < na ? d : na;
    while (lo < hi) {
        const uint64_t span = hi - lo;
        const uint32_t c = count(lo, span, d);
        if (span <= 64) return lo + c;
        const uint64_t nlo = c ? merge_probe(lo, span, c - 1) + 1 : lo, nhi = c < 64 ? merge_probe(lo, span, c) : hi;
        lo = nlo;
        hi = nhi;
    }
    return lo;
}

struct merge_part {
    uint64_t a0, b0;    // where the tile's values begin in a and b
    uint32_t la, lb;    // how many of each it takes
};

// The part of the places [d0, d1) of the merged order whose splits are s0
// and s1 (of merge_split).  The two come from searches of their own: with
// lists that are not ascending s1 may lie below s0 or further from it than
// d1 - d0, so the part is cut to the lists and to the tile.
__host__ __device__ __forceinline__ merge_part merge_part_of(uint64_t s0, uint64_t s1, uint64_t d0, uint64_t d1,
                                                             uint64_t na, uint64_t nb)
{
    const uint64_t len = d1 - d0;
    merge_part p;
    p.a0 = s0;
    p.b0 = d0 - s0;
    const uint64_t end = s0 + len < na ? s0 + len : na;
    const uint64_t a1 = s1 < s0 ? s0 : s1 < end ? s1 : end;
    p.la = (uint32_t)(a1 - s0);
    const uint64_t lb = len - p.la;
    p.lb = (uint32_t)(lb < nb - p.b0 ? lb : nb - p.b0);
    return p;
}

}  // namespace ms
