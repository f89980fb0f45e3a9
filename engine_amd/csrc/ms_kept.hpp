// ms_kept.hpp -- device memory of the null stream, kept for its next call.
//
// hipMallocAsync's pool gives memory back to the system on a free whatever
// its release threshold says, so that every call maps and unmaps its buffers
// again: of the select, project and agg_sum over 2^24 values (0.31 ms of
// kernels) that was 0.8 to 12 ms, growing with the memory the process holds.
// A block freed on the null stream is handed to a later call on the null
// stream without waiting: the stream orders its uses, and unlike a created
// stream it is never destroyed and never captured; created streams, which it
// waits for, may read a block until then; other streams keep
// using hipMallocAsync.  At most a sixteenth of a device's memory is kept (the
// least recently freed blocks go first).
//
// Nothing here throws: the entry points that allocate are C.
//
// The rules only: `Api` is the device's side, so that they can be checked on
// the host.  It has static device() (the current one), alloc(device, bytes),
// free(device, p), settle(device) (waits for the device and gives its unused
// memory to the system) and total(device) (its bytes).
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <deque>
#include <iterator>
#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>

namespace ms {

template <class Api>
class kept_memory {
    struct block {
        void *p;
        size_t bytes;
        int dev;
        size_t over;   // bytes more than its use asks for
    };
    typedef std::list<block> lru;                            // free blocks, least recently freed first
    struct device {
        lru free_;
        // blocks of each size, least recently freed first as well: get()
        // takes a class's last one, trim() the first of the one it is in
        std::map<size_t, std::deque<typename lru::iterator>> by_size;
        size_t kept = 0, limit = 0, over = 0;   // over: of all blocks in use
    };
    static constexpr int MAX_DEVICES = 64;
    // A block may be a quarter larger than asked for, but a column holds it
    // for as long as it lives: all blocks in use together are at most this
    // much too large.
    static constexpr size_t MAX_OVER = 64u << 20;

    std::mutex mu;
    std::unordered_map<void *, block> live;                  // blocks in use
    device devs[MAX_DEVICES];

    // Sizes are rounded up to what the pool takes from the system for them
    // anyway (pages of 4 KiB up to 1 MiB, of 2 MiB above), so that calls of
    // nearly the same sizes share blocks and no memory is lost.
    static size_t round_size(size_t n)
    {
        const size_t page = n <= (1u << 20) ? 4096 : 2u << 20;
        return n > SIZE_MAX - page ? n : (n + page - 1) / page * page;
    }

    typedef typename std::map<size_t, std::deque<typename lru::iterator>>::iterator size_class;

    // Takes the last or the first block of a size class out of the lists.
    static block take(device &d, size_class b, bool last)
    {
        const auto it = last ? b->second.back() : b->second.front();
        const block k = *it;
        if (last) b->second.pop_back();
        else b->second.pop_front();
        if (b->second.empty()) d.by_size.erase(b);
        d.kept -= k.bytes;
        d.free_.erase(it);
        return k;
    }

    static void trim(device &d, size_t to)
    {
        while (d.kept > to && !d.free_.empty()) {
            const block k = take(d, d.by_size.find(d.free_.front().bytes), false);
            Api::free(k.dev, k.p);
        }
    }

    void give_back(int dev)
    {
        if (devs[dev].free_.empty()) return;
        trim(devs[dev], 0);
        Api::settle(dev);
    }

    // Notes a block in use and gives its address.  Without host memory for
    // that the caller has it all the same: put() then does not know it.
    void *hold(const block &k)
    {
        try {
            live.emplace(k.p, k);
        } catch (...) {
            devs[k.dev].over -= k.over;
        }
        return k.p;
    }

public:
    // Memory of the current device for a call on the null stream.
    void *get(size_t bytes)
    {
        const int dev = Api::device();
        if (dev < 0 || dev >= MAX_DEVICES) return nullptr;
        const size_t want = round_size(bytes);
        std::lock_guard<std::mutex> lk(mu);
        device &d = devs[dev];
        // the smallest block that fits, unless it is too large
        auto b = d.by_size.lower_bound(want);
        if (b != d.by_size.end() && b->first - want <= want / 4 && d.over + (b->first - want) <= MAX_OVER) {
            block k = take(d, b, true);
            k.over = k.bytes - want;
            d.over += k.over;
            return hold(k);
        }
        block k = {Api::alloc(dev, want), want, dev, 0};
        if (!k.p) {
            give_back(dev);
            k.p = Api::alloc(dev, want);
            if (!k.p) return nullptr;
        }
        return hold(k);
    }

    // Takes back memory of get(), whatever device is current; `keep` false:
    // to the pool, not for a later call.  false: not a block of this object.
    bool put(void *p, bool keep = true)
    {
        std::lock_guard<std::mutex> lk(mu);
        auto l = live.find(p);
        if (l == live.end()) return false;
        const block k = l->second;
        live.erase(l);
        device &d = devs[k.dev];
        d.over -= k.over;
        if (!d.limit) {
            const size_t total = Api::total(k.dev);
            d.limit = total ? total / 16 : 1u << 30;
        }
        if (!keep || k.bytes > d.limit) {
            Api::free(k.dev, p);
            return true;
        }
        try {
            d.free_.push_back(k);
            try {
                d.by_size[k.bytes].push_back(std::prev(d.free_.end()));
            } catch (...) {
                const auto b = d.by_size.find(k.bytes);
                if (b != d.by_size.end() && b->second.empty()) d.by_size.erase(b);
                d.free_.pop_back();
                throw;
            }
        } catch (...) {   // no host memory to keep it with
            Api::free(k.dev, p);
            return true;
        }
        d.kept += k.bytes;
        trim(d, d.limit);
        return true;
    }

    // Frees every block that is not in use.
    void drop()
    {
        std::lock_guard<std::mutex> lk(mu);
        for (device &d : devs) trim(d, 0);
    }

    // The same, and everything unused goes to the system.
    void release()
    {
        std::lock_guard<std::mutex> lk(mu);
        for (int dev = 0; dev < MAX_DEVICES; dev++) give_back(dev);
    }
};

}  // namespace ms
