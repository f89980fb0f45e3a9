// merge_sorted's tile arithmetic (engine_amd/csrc/ms_merge_path.hpp) on the
// host: every tile's part of lists in any order lies inside both lists and
// inside the tile, and of ascending lists the parts are the merge path's.
#include <stdint.h>
#include <stdio.h>

#include <algorithm>
#include <numeric>
#include <random>
#include <vector>

#include "ms_merge_path.hpp"

typedef std::vector<uint64_t> list;
static int g_bad = 0;

#define CHECK(cond, ...)                                                      \
    do {                                                                      \
        if (!(cond) && g_bad++ < 20) {                                        \
            printf("%s:%d: %s: ", __FILE__, __LINE__, #cond);                 \
            printf(__VA_ARGS__);                                              \
            printf("\n");                                                     \
        }                                                                     \
    } while (0)

// what the 64 lanes of a wave count
struct host_count {
    const list &a, &b;
    uint32_t operator()(uint64_t lo, uint64_t span, uint64_t d) const
    {
        uint32_t c = 0;
        for (uint32_t t = 0; t < 64; t++) {
            const uint64_t i = ms::merge_probe(lo, span, t);
            if (i >= lo + span) continue;
            CHECK(i < a.size() && d - 1 - i < b.size(), "probe %llu of %llu", (unsigned long long)i, (unsigned long long)d);
            if (i < a.size() && d - 1 - i < b.size()) c += a[i] <= b[d - 1 - i];
        }
        return c;
    }
};

static void lists(const char *name, const list &a, const list &b, uint64_t tile)
{
    const uint64_t na = a.size(), nb = b.size(), n = na + nb;
    const bool ascending = std::is_sorted(a.begin(), a.end()) && std::is_sorted(b.begin(), b.end());
    for (uint64_t d0 = 0; d0 < n; d0 += tile) {
        const uint64_t d1 = std::min(d0 + tile, n);
        const uint64_t s0 = ms::merge_split(na, nb, d0, host_count{a, b});
        const uint64_t s1 = ms::merge_split(na, nb, d1, host_count{a, b});
        CHECK(s0 <= std::min(d0, na) && d0 - s0 <= nb, "%s at %llu", name, (unsigned long long)d0);
        const ms::merge_part p = ms::merge_part_of(s0, s1, d0, d1, na, nb);
        CHECK(p.a0 + p.la <= na && p.b0 + p.lb <= nb && (uint64_t)p.la + p.lb <= d1 - d0, "%s at %llu: %u of a from %llu, %u of b from %llu",
              name, (unsigned long long)d0, p.la, (unsigned long long)p.a0, p.lb, (unsigned long long)p.b0);
        if (!ascending) continue;
        CHECK((uint64_t)p.la + p.lb == d1 - d0 && p.a0 + p.la == s1, "%s at %llu", name, (unsigned long long)d0);
        // a first among equals: what lies before the split is below what lies behind
        CHECK(s0 == 0 || d0 - s0 == nb || a[s0 - 1] <= b[d0 - s0], "%s at %llu", name, (unsigned long long)d0);
        CHECK(s0 == na || d0 == s0 || b[d0 - s0 - 1] < a[s0], "%s at %llu", name, (unsigned long long)d0);
    }
}

int main()
{
    std::mt19937_64 rng(1);
    const auto uniform = [&](uint64_t n, uint64_t below) {
        list v(n);
        for (uint64_t &x : v) x = rng() % below;
        return v;
    };
    const auto sorted = [](list v) {
        std::sort(v.begin(), v.end());
        return v;
    };
    const uint64_t T = 8192;
    // a part of negative size without the cut: splits 8192 and 4096
    list a(T, 1), b(T, 1);
    a.insert(a.end(), 4096, 5);
    b.insert(b.end(), 4096, 0);
    lists("ones then 5 / ones then 0", a, b, T);
    for (uint64_t na : {0, 1, 64, 65, 4097, 8192, 100000})
        for (uint64_t nb : {0, 1, 63, 8191, 50000})
            for (uint64_t below : {2ull, 1000ull, 1ull << 40}) {
                const list x = uniform(na, below), y = uniform(nb, below);
                for (uint64_t tile : {T, (uint64_t)96}) {
                    lists("ascending", sorted(x), sorted(y), tile);
                    lists("shuffled", x, y, tile);
                    lists("ascending / shuffled", sorted(x), y, tile);
                    lists("shuffled / ascending", x, sorted(y), tile);
                }
            }
    list up(100000), down(100000);
    std::iota(up.begin(), up.end(), 0);
    std::iota(down.rbegin(), down.rend(), 0);
    lists("up / down", up, down, T);
    lists("down / up", down, up, T);
    if (g_bad) return printf("%d checks failed\n", g_bad), 1;
    printf("merge path ok\n");
    return 0;
}
