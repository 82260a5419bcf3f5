// hss_pool.h -- device memory that comes and goes with every `\`: factors, their workspace,
// plans, host-call buffers.  No HIP here: Mem::alloc(bytes) (null when there is none) and
// Mem::release(p) are the device's.  Not part of the public ABI.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <map>
#include <mutex>
#include <new>
#include <utility>
#include <vector>

namespace hss {

// Blocks given back are kept for the next request of about their size, up to kHeldMax bytes
// and kHeldBlocks blocks, the oldest freed first.  They are all freed with the pool, by trim(), and
// whenever an allocation on the device fails (allocate(), for every allocation of the library),
// so that what is held never keeps something else from fitting.  hipMalloc and hipFree cost
// tens to hundreds of microseconds each (mapping and unmapping).
// A new block is rounded up by at most a sixteenth, and a held one is taken up to an eighth
// above that, so that matrices with slightly other ranks share blocks; `exact` asks for the
// request and no more (in pages), which is what a block kept for long gets.  *got is the size handed
// out.
template <class Mem>
class BlockPool {
public:
    BlockPool() = default;
    BlockPool(const BlockPool&) = delete;
    BlockPool& operator=(const BlockPool&) = delete;
    ~BlockPool() {
        detach();
        trim();
    }

    // its held blocks count as free memory of `device` from here on
    void attach(int device) {
        detach();
        std::lock_guard<std::mutex> lk(registry().mu);
        registry().pools.emplace_back(device, this);
    }
    void detach() {
        std::lock_guard<std::mutex> lk(registry().mu);
        auto& v = registry().pools;
        v.erase(std::remove_if(v.begin(), v.end(), [&](const auto& e) { return e.second == this; }), v.end());
    }

    // Mem::alloc; on failure once more after every pool of the device has freed what it holds
    static void* allocate(int device, size_t bytes) noexcept {
        void* p = Mem::alloc(bytes);
        if (p) return p;
        bool freed = false;
        {
            std::lock_guard<std::mutex> lk(registry().mu);
            for (auto& e : registry().pools)
                if (e.first == device) freed |= e.second->trim();
        }
        return freed ? Mem::alloc(bytes) : nullptr;
    }

    static size_t rounded(size_t bytes, bool exact) {
        size_t step = kPage;
        if (!exact)
            while (32 * step <= bytes) step *= 2;
        return (std::max<size_t>(bytes, 1) + step - 1) / step * step;
    }

    // null: out of memory (of the device or, for the bookkeeping, of the host)
    void* get(int device, size_t bytes, bool exact = false, size_t* got = nullptr) noexcept {
        size_t size = rounded(bytes, exact);
        {
            std::lock_guard<std::mutex> lk(mu);
            const auto it = held.lower_bound(size);
            if (it != held.end() && it->first <= (exact ? size : size + size / 8)) {
                void* p = it->second.p;
                size = it->first;
                if (!note(p, size)) return nullptr;
                held_bytes -= size;
                held.erase(it);
                if (got) *got = size;
                return p;
            }
        }
        void* p = allocate(device, size);
        if (!p && !exact) p = allocate(device, size = rounded(bytes, true));  // the last of the memory
        if (!p) return nullptr;
        std::lock_guard<std::mutex> lk(mu);
        if (!note(p, size)) {
            Mem::release(p);
            return nullptr;
        }
        if (got) *got = size;
        return p;
    }

    // p from get(); nothing may still use it
    void put(void* p) noexcept {
        if (!p) return;
        std::lock_guard<std::mutex> lk(mu);
        const auto u = used.find(p);
        const size_t bytes = u->second;
        used.erase(u);
        if (bytes > kHeldMax) {
            Mem::release(p);
            return;
        }
        while (held_bytes + bytes > kHeldMax || held.size() >= kHeldBlocks) drop_oldest();
        try {
            held.emplace(bytes, Held{p, ++clock});
            held_bytes += bytes;
        } catch (const std::bad_alloc&) {
            Mem::release(p);
        }
    }

    // frees the held blocks; true if there were any
    bool trim() noexcept {
        std::lock_guard<std::mutex> lk(mu);
        const bool any = !held.empty();
        for (auto& h : held) Mem::release(h.second.p);
        held.clear();
        held_bytes = 0;
        return any;
    }

    static constexpr size_t kPage = 4096, kHeldMax = size_t(2) << 30, kHeldBlocks = 512;

private:
    struct Held {
        void* p;
        uint64_t age;
    };
    struct Registry {
        std::mutex mu;  // taken before a pool's own
        std::vector<std::pair<int, BlockPool*>> pools;
    };
    static Registry& registry() {
        static auto* r = new Registry;  // outlives every static object that holds a pool
        return *r;
    }
    bool note(void* p, size_t bytes) noexcept {
        try {
            used.emplace(p, bytes);
            return true;
        } catch (const std::bad_alloc&) {
            return false;
        }
    }
    void drop_oldest() noexcept {
        auto old = held.begin();
        for (auto it = held.begin(); it != held.end(); ++it)
            if (it->second.age < old->second.age) old = it;
        Mem::release(old->second.p);
        held_bytes -= old->first;
        held.erase(old);
    }
    std::mutex mu;
    std::multimap<size_t, Held> held;  // by size
    std::map<void*, size_t> used;
    size_t held_bytes = 0;
    uint64_t clock = 0;
};

}  // namespace hss
