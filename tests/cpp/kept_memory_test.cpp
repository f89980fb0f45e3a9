// The rules of the null stream's kept memory (engine_amd/csrc/ms_kept.hpp) on
// the host, over devices that are only counted.  argv[1] names the check.
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <map>
#include <new>
#include <vector>

#include "ms_kept.hpp"

#define CHECK(cond)                                                           \
    do {                                                                      \
        if (!(cond)) {                                                        \
            printf("%s:%d: %s\n", __FILE__, __LINE__, #cond);                 \
            exit(1);                                                          \
        }                                                                     \
    } while (0)

static const size_t MiB = 1u << 20;

// operator new fails from the g_news-th call on, for g_fails calls.
static long g_news = -1, g_fails = 0;
__attribute__((noinline)) void *operator new(size_t n)
{
    if (g_news == 0 && g_fails > 0) {
        g_fails--;
        throw std::bad_alloc();
    }
    if (g_news > 0) g_news--;
    if (void *p = malloc(n)) return p;
    throw std::bad_alloc();
}
__attribute__((noinline)) void operator delete(void *p) noexcept { free(p); }
__attribute__((noinline)) void operator delete(void *p, size_t) noexcept { free(p); }
struct host_memory_back {                     // for the test's own bookkeeping
    long news = g_news;
    host_memory_back() { g_news = -1; }
    ~host_memory_back() { g_news = news; }
};

// Two devices of `size` bytes; an allocation is a key of `held`.
struct fake {
    struct mem {
        int dev;
        size_t bytes;
    };
    static std::map<void *, mem> held;
    static size_t size, used[2];
    static int current, settled[2], frees;
    static uintptr_t next;

    static int device() { return current; }
    static void *alloc(int dev, size_t bytes)
    {
        const host_memory_back ours;
        CHECK(dev == current && bytes);
        if (used[dev] + bytes > size) return nullptr;
        void *p = (void *)next;
        next += 256;
        held[p] = mem{dev, bytes};
        used[dev] += bytes;
        return p;
    }
    static void free(int dev, void *p)
    {
        auto h = held.find(p);
        CHECK(h != held.end() && h->second.dev == dev);   // freed under its own device
        used[dev] -= h->second.bytes;
        held.erase(h);
        frees++;
    }
    static void settle(int dev) { settled[dev]++; }
    static size_t total(int dev) { return size / (1 + dev); }
};
std::map<void *, fake::mem> fake::held;
size_t fake::size = 1024 * MiB, fake::used[2];
int fake::current, fake::settled[2], fake::frees;
uintptr_t fake::next = 4096;

typedef ms::kept_memory<fake> kept;

static void reuse(kept &k)
{
    void *a = k.get(MiB), *b = k.get(3 * MiB);
    CHECK(a && b && a != b && fake::held[a].bytes >= MiB);
    CHECK(!k.put((void *)8));                 // not its block
    CHECK(k.put(a) && !k.put(a));             // once only
    CHECK(k.get(MiB) == a);                   // handed out again
    void *c = k.get(MiB);
    CHECK(c != a && c != b);                  // never to two calls
    CHECK(k.put(b) && k.get(MiB) != b);       // far too large
    CHECK(fake::frees == 0);
    CHECK(k.put(c, false) && !fake::held.count(c) && fake::frees == 1);   // not to be kept
}

// A sixteenth of the device is kept; the least recently freed goes first.
static void limit(kept &k)
{
    void *p[40];
    for (int i = 0; i < 40; i++) p[i] = k.get(4 * MiB);
    void *large = k.get(65 * MiB);
    for (int i = 0; i < 16; i++) CHECK(k.put(p[i]));
    CHECK(fake::frees == 0);
    for (int i = 16; i < 19; i++) {
        CHECK(k.put(p[i]) && fake::held.count(p[i]));
        CHECK(!fake::held.count(p[i - 16]));
    }
    CHECK(fake::frees == 3);
    CHECK(k.put(large) && !fake::held.count(large) && fake::frees == 4);   // above the limit by itself
    CHECK(k.get(4 * MiB) == p[18]);           // the latest, warm in the caches
}

static void failure(kept &k)
{
    void *a = k.get(40 * MiB), *b = k.get(896 * MiB);
    CHECK(a && b && k.put(a));
    void *c = k.get(96 * MiB);                // does not fit beside the kept block
    CHECK(c && !fake::held.count(a) && fake::settled[0] == 1);
    CHECK(k.get(96 * MiB) == nullptr && fake::settled[0] == 1);   // nothing left to give back
    CHECK(k.put(c) && k.put(b));
}

static void drop(kept &k)
{
    void *a = k.get(MiB), *b = k.get(2 * MiB);
    CHECK(k.put(a));
    k.drop();
    CHECK(!fake::held.count(a) && fake::held.count(b) && fake::settled[0] == 0);
    CHECK(k.put(b));
    k.release();
    CHECK(fake::held.empty() && fake::settled[0] == 1);
}

// Blocks stay with their device: reuse, frees, limits, give-back.
static void devices(kept &k)
{
    void *a = k.get(MiB), *a2 = k.get(2 * MiB);
    fake::current = 1;
    void *b = k.get(MiB), *b2 = k.get(2 * MiB);
    CHECK(k.put(a) && k.put(b));              // a's device is not the current one
    CHECK(k.get(MiB) == b);
    fake::current = 0;
    CHECK(k.get(MiB) == a);
    CHECK(k.put(a) && k.put(a2) && k.put(b) && k.put(b2));
    void *p[20];
    for (int i = 0; i < 20; i++) p[i] = k.get(4 * MiB);
    for (int i = 0; i < 20; i++) k.put(p[i]);  // device 0's limit
    CHECK(fake::used[0] <= 64 * MiB && fake::used[0] >= 56 * MiB && fake::held.count(b) && fake::held.count(b2));
    fake::current = 1;
    for (int i = 0; i < 20; i++) p[i] = k.get(4 * MiB);
    for (int i = 0; i < 20; i++) k.put(p[i]);  // half as large
    CHECK(fake::used[1] <= 32 * MiB && fake::used[1] >= 24 * MiB && fake::used[0] >= 56 * MiB);
    void *big = k.get(1000 * MiB);            // fits once device 1's blocks are gone
    CHECK(big && fake::settled[1] == 1 && fake::settled[0] == 0 && fake::used[0] >= 56 * MiB);
    k.drop();
    CHECK(fake::used[0] == 0);
}

// Finding and freeing a block takes no longer the more of its size are free.
static void many(kept &k)
{
    const int n = 500000;
    fake::size = (size_t)n * 4096 * 32;
    std::vector<void *> p(n);
    for (int i = 0; i < n; i++) p[i] = k.get(1000);
    for (int i = 0; i < n; i++) CHECK(k.put(p[i]));
    CHECK(fake::frees == 0);
    for (int i = 0; i < n; i++) CHECK(k.get(1000) == p[n - 1 - i]);   // the latest first
    for (int i = 0; i < n; i++) CHECK(k.put(p[i]));
    k.drop();
    CHECK(fake::frees == n);
}

// What fits without the cache fits with it: a block is larger than asked for
// by less than the pool's page, and larger ones are reused within a budget.
static void excess(kept &k)
{
    for (size_t n : {(size_t)1, (size_t)4096, (size_t)5000, MiB, MiB + 1, 3 * MiB + 256, 33 * MiB + 256, 700 * MiB + 1}) {
        void *p = k.get(n);
        CHECK(p && fake::held[p].bytes >= n && fake::held[p].bytes - n < (n <= MiB ? 4096 : 2 * MiB));
        CHECK(k.put(p));
        k.drop();
    }
    void *a = k.get(901 * MiB), *b = k.get(121 * MiB);
    CHECK(a && b && k.put(a) && k.put(b));
    k.drop();
    CHECK(k.get(SIZE_MAX - 100) == nullptr && k.get(SIZE_MAX) == nullptr);

    fake::size = 64 * 1024 * MiB;             // 4 GiB are kept
    kept l;
    void *p[10], *q[10];
    for (void *&x : p) x = l.get(120 * MiB);
    for (void *x : p) CHECK(l.put(x));
    for (int i = 0; i < 10; i++) {
        q[i] = l.get(100 * MiB);              // 20 MiB too large, three times
        CHECK((fake::held[q[i]].bytes == 120 * MiB) == (i < 3));
    }
    CHECK(l.put(q[1]));
    void *r = l.get(101 * MiB);               // the budget is free again
    CHECK(fake::held[r].bytes == 120 * MiB);
    CHECK(l.get(80 * MiB) && fake::held.size() == 10 + 7 + 1);   // 40 MiB too large: never
}

// Without host memory calls are served and nothing is lost or freed twice:
// one to three allocations of the host fail at every point of a few calls.
static void host_memory(kept &)
{
    for (long fails = 1; fails <= 3; fails++)
        for (long at = 0; at < 40; at++) {
            kept k;
            void *p[6];
            for (int round = 0; round < 3; round++) {
                if (round == 1) {
                    g_news = at;
                    g_fails = fails;
                }
                for (int i = 0; i < 6; i++) {
                    p[i] = k.get((1 + i / 2) * 8192);
                    CHECK(p[i] && fake::held.count(p[i]));
                    for (int j = 0; j < i; j++) CHECK(p[j] != p[i]);
                }
                for (int i = 0; i < 6; i++)
                    if (!k.put(p[i])) fake::free(0, p[i]);   // as the caller does
            }
            g_news = -1;
            CHECK(k.get(8192));
            k.drop();
            CHECK(fake::held.size() == 1);
            fake::free(0, fake::held.begin()->first);
        }
}

int main(int argc, char **argv)
{
    const std::pair<const char *, void (*)(kept &)> checks[] = {
        {"reuse", reuse}, {"limit", limit}, {"failure", failure}, {"drop", drop}, {"devices", devices},
        {"many", many}, {"excess", excess},
        {"host_memory", host_memory}};
    for (const auto &c : checks)
        if (argc > 1 && !strcmp(argv[1], c.first)) {
            kept k;
            c.second(k);
            printf("%s ok\n", c.first);
            return 0;
        }
    return 2;
}
