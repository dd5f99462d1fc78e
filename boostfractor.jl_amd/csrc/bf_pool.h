// bf_pool.h -- device memory of a context: owning buffers and the blocks kept between them.
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "../../include/boostfractor_hip.h"

namespace bf {

// Internal failure carrying a C-ABI status code; converted to a return code at
// the extern "C" boundary.
struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

// Device memory given back by the buffers of one context, for its next ones.  A call
// allocates a dozen buffers and frees them when it returns; hipMalloc and hipFree take
// ~9 us each (milliseconds for hundreds of MB, and hipFree waits for the device).
// Everything a context does is ordered on its one stream, so memory that work queued
// earlier may still use can be handed out again at once.  The pool keeps at most
// `keep` bytes (the last ones given back; option pool_mb), and frees them all when an
// allocation of any context on its device fails and when its context is destroyed;
// blocks that come back later are freed directly.  A plan may be destroyed on another
// thread than its context's calls, and another context's thread may free what is kept
// here: the lock.  (hipFree waits for the device, so for the work that still uses it.)
class DevPool {
  public:
    static constexpr size_t KEEP = (size_t)2 << 30;
    explicit DevPool(int dev = 0) : device(dev) {
        Registry& r = registry();
        std::lock_guard<std::mutex> lk(r.mu);
        r.pools.push_back(this);
    }
    DevPool(const DevPool&) = delete;
    DevPool& operator=(const DevPool&) = delete;
    ~DevPool() {
        {
            Registry& r = registry();
            std::lock_guard<std::mutex> lk(r.mu);
            r.pools.erase(std::find(r.pools.begin(), r.pools.end(), this));
        }
        trim(true);
    }
    // block sizes: multiples of an eighth of the next lower power of two (at least 512 bytes)
    static size_t round(size_t n) {
        size_t g = 512;
        while (g * 16 <= n) g *= 2;
        return (n + g - 1) / g * g;
    }
    void* take(size_t block) {
        std::lock_guard<std::mutex> lk(mu);
        auto it = blocks.find(block);
        if (it == blocks.end()) return nullptr;
        void* p = it->second.first;
        blocks.erase(it);
        kept -= block;
        return p;
    }
    // (called from destructors: a block that cannot be entered is freed)
    void give(void* p, size_t block) noexcept {
        bool entered = false;
        try {
            std::lock_guard<std::mutex> lk(mu);
            if (!closed && block <= keep) {
                blocks.emplace(block, std::make_pair(p, ++turn));
                kept += block;
                entered = true;
            }
        } catch (...) {
        }
        if (!entered) (void)hipFree(p);
        shrink();
    }
    // most bytes to keep from now on
    void limit(size_t bytes) noexcept {
        {
            std::lock_guard<std::mutex> lk(mu);
            keep = bytes;
        }
        shrink();
    }
    void trim(bool close = false) noexcept {
        decltype(blocks) out;
        {
            std::lock_guard<std::mutex> lk(mu);
            out.swap(blocks);
            kept = 0;
            closed = closed || close;
        }
        for (auto& b : out) (void)hipFree(b.second.first);
    }
    // frees what the contexts of a device keep
    static void trim_all(int dev) noexcept {
        Registry& r = registry();
        std::lock_guard<std::mutex> lk(r.mu);
        for (DevPool* p : r.pools)
            if (p->device == dev) p->trim();
    }
    void on_device(int dev) { device = dev; }  // before the context's first call

  private:
    struct Registry {
        std::mutex mu;
        std::vector<DevPool*> pools;
    };
    // never destroyed: contexts may outlive the library's static objects
    static Registry& registry() {
        static Registry* r = new Registry();
        return *r;
    }
    // the blocks that lay unused longest go until the rest is within the limit
    void shrink() noexcept {
        for (;;) {
            void* p = nullptr;
            {
                std::lock_guard<std::mutex> lk(mu);
                if (kept <= keep) return;
                auto old = std::min_element(blocks.begin(), blocks.end(), [](const auto& a, const auto& b) {
                    return a.second.second < b.second.second;
                });
                p = old->second.first;
                kept -= old->first;
                blocks.erase(old);
            }
            (void)hipFree(p);
        }
    }
    std::mutex mu;
    std::multimap<size_t, std::pair<void*, uint64_t>> blocks;  // by size: address, turn it came back
    size_t kept = 0, keep = KEEP;
    uint64_t turn = 0;
    bool closed = false;
    int device;
};
// pool of the context whose call runs on this thread (null outside a call)
const std::shared_ptr<DevPool>& call_pool();

// Owning device allocation.
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    explicit DevBuf(size_t n) { alloc(n); }
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    DevBuf(DevBuf&& o) noexcept : p(o.p), bytes(o.bytes), block(o.block), pool(std::move(o.pool)) {
        o.p = nullptr;
        o.bytes = 0;
    }
    DevBuf& operator=(DevBuf&& o) noexcept {
        if (this != &o) {
            release();
            p = o.p;
            bytes = o.bytes;
            block = o.block;
            pool = std::move(o.pool);
            o.p = nullptr;
            o.bytes = 0;
        }
        return *this;
    }
    ~DevBuf() { release(); }
    void alloc(size_t n) {
        release();
        if (n == 0) return;
        pool = call_pool();
        block = pool ? DevPool::round(n) : n;
        if (pool) p = pool->take(block);
        if (!p) {
            hipError_t e = hipMalloc(&p, block);
            if (e == hipErrorOutOfMemory) {  // what the pools keep, and the rounding, may be what is missing
                (void)hipGetLastError();
                int dev = 0;
                (void)hipGetDevice(&dev);
                DevPool::trim_all(dev);
                block = n;
                e = hipMalloc(&p, block);
            }
            if (e != hipSuccess) {
                p = nullptr;
                pool.reset();
                throw Error(e == hipErrorOutOfMemory ? BF_ERR_NOMEM : BF_ERR_HIP,
                            std::string("hipMalloc(") + std::to_string(n) + " bytes): " + hipGetErrorString(e));
            }
        }
        bytes = n;
    }
    void release() {
        if (p) {
            if (pool)
                pool->give(p, block);
            else
                (void)hipFree(p);
        }
        p = nullptr;
        bytes = 0;
        pool.reset();
    }
    template <typename U>
    U* as() const { return static_cast<U*>(p); }

  private:
    size_t block = 0;  // bytes allocated
    std::shared_ptr<DevPool> pool;
};

}  // namespace bf
