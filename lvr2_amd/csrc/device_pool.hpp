// Device memory of destroyed handles and finished host calls, kept for the next ones.
//
// hipMalloc and hipFree dominated short jobs: a surface of 500,000 points made and freed for one normals
// pass spent 3.6 ms in its frees and 1 ms in its allocations beside 7 ms of kernels.  A freed block goes to
// a list of its device and size class instead and serves the next allocation of that class.
//  - Safe across streams and threads: a block enters the list only from a scope that has waited for the
//    device's work on it (IdleScope); freed anywhere else it goes back to the runtime.  One mutex
//    guards the lists.
//  - Bounded: at most CACHE_BYTES per device, no block above a quarter of that.
//  - Given back: blocks that no allocation took over the last KEEP calls that return blocks (host-array calls and
//    handle destructions, on any device) are freed, all of a device's blocks when one of its
//    allocations fails (which is then tried again), and all there are by release() (lvrhip_release_memory).
//    Not with the last handle: one surface after the other, each destroyed before the next, is what the
//    pool is for.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <map>
#include <mutex>
#include <unordered_map>
#include <utility>
#include <vector>

namespace lvrhip {

class DevicePool {
public:
    static constexpr size_t CACHE_BYTES = (size_t)2 << 30;
    static constexpr size_t KEPT_BLOCK = CACHE_BYTES / 4;  // the largest block kept
    static constexpr uint64_t KEEP = 64;
    static constexpr size_t PINNED_BYTES = 64;
    static constexpr size_t PINNED_KEPT = 64;
    static constexpr int ALL = -1;

    static DevicePool& get()
    {
        static DevicePool* p = new DevicePool;  // never destroyed: handles may outlive static destructors
        return *p;
    }

    // a block of at least `bytes` on the current device
    hipError_t alloc(void** p, size_t bytes)
    {
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return e;
        const size_t size = size_class(bytes);
        {
            std::lock_guard<std::mutex> lk(mu_);
            auto& c = cache_[dev];
            auto it = c.blocks.find(size);
            if (it != c.blocks.end() && !it->second.empty()) {
                live_[it->second.back().first] = {dev, size};
                *p = it->second.back().first;
                it->second.pop_back();
                c.bytes -= size;
                return hipSuccess;
            }
        }
        size_t got = size;
        e = hipMalloc(p, size);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();
            trim(dev, ~0ull);
            got = bytes;
            e = hipMalloc(p, bytes);
        }
        if (e != hipSuccess) return e;
        try {
            std::lock_guard<std::mutex> lk(mu_);
            live_[*p] = {dev, got};
        } catch (...) {
            (void)hipFree(*p);
            throw;
        }
        return hipSuccess;
    }

    // idle: no work of any stream on the block is left.  Runs in destructors: a block that the lists have no host
    // memory for goes back to the runtime.
    void free(void* p, bool idle) noexcept
    {
        bool keep = false;
        try {
            std::lock_guard<std::mutex> lk(mu_);
            auto it = live_.find(p);
            if (it != live_.end()) {
                const auto [dev, size] = it->second;
                live_.erase(it);
                auto& c = cache_[dev];
                if (idle && size == size_class(size) && size <= KEPT_BLOCK && c.bytes + size <= CACHE_BYTES) {
                    c.blocks[size].emplace_back(p, now_);
                    c.bytes += size;
                    keep = true;
                }
            }
        } catch (...) {
        }
        if (!keep) (void)hipFree(p);
    }

    // a call returned its blocks: what nobody took for KEEP of these is freed
    void tick() noexcept
    {
        uint64_t t;
        {
            std::lock_guard<std::mutex> lk(mu_);
            t = ++now_;
        }
        if (t > KEEP) trim(ALL, t - KEEP);
    }

    // frees all that is kept for a device (ALL: for every one); returns the bytes
    size_t release(int dev) noexcept { return trim(dev, ~0ull); }

    // pinned host words for readbacks
    hipError_t alloc_pinned(uint32_t** p)
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            if (!pinned_.empty()) {
                *p = pinned_.back();
                pinned_.pop_back();
                return hipSuccess;
            }
        }
        return hipHostMalloc(reinterpret_cast<void**>(p), PINNED_BYTES, hipHostMallocPortable);
    }
    void free_pinned(uint32_t* p, bool idle) noexcept
    {
        try {
            std::lock_guard<std::mutex> lk(mu_);
            if (idle && pinned_.size() < PINNED_KEPT) {
                pinned_.push_back(p);
                return;
            }
        } catch (...) {
        }
        (void)hipHostFree(p);
    }

private:
    struct Cache {
        std::map<size_t, std::vector<std::pair<void*, uint64_t>>> blocks;  // by size: (block, when freed)
        size_t bytes = 0;
    };
    std::mutex mu_;
    std::map<int, Cache> cache_;
    std::unordered_map<void*, std::pair<int, size_t>> live_;
    std::vector<uint32_t*> pinned_;
    uint64_t now_ = 0;

    // sizes in steps of an eighth of the power of two below (at most 12.5 % more than asked for); a block too
    // large to be kept has just the size asked for
    static size_t size_class(size_t bytes)
    {
        if (bytes <= 4096) return 4096;
        if (bytes > KEPT_BLOCK) return bytes;
        const size_t step = ((size_t)1 << (63 - __builtin_clzll(bytes))) / 8;
        return (bytes + step - 1) / step * step;
    }

    // frees the kept blocks of a device (ALL: of every one) that were freed before `before`; returns the bytes
    size_t trim(int dev, uint64_t before) noexcept
    {
        size_t bytes = 0;
        while (void* p = take_kept(dev, before, bytes)) (void)hipFree(p);
        return bytes;
    }
    void* take_kept(int dev, uint64_t before, size_t& bytes) noexcept
    {
        std::lock_guard<std::mutex> lk(mu_);
        for (auto& [d, c] : cache_) {
            if (dev != ALL && d != dev) continue;
            for (auto& [size, v] : c.blocks) {
                for (auto& b : v) {
                    if (b.second >= before) continue;
                    void* p = b.first;
                    b = v.back();
                    v.pop_back();
                    c.bytes -= size;
                    bytes += size;
                    return p;
                }
            }
        }
        return nullptr;
    }
};

// While one is set on a thread, the blocks that the thread frees are known to be idle: set it after waiting
// for all work on them.  Its end is a call's end for the pool (tick).
struct IdleScope {
    bool on = false;
    static bool& flag()
    {
        static thread_local bool f = false;
        return f;
    }
    void set()
    {
        on = true;
        flag() = true;
    }
    ~IdleScope()
    {
        if (!on) return;
        flag() = false;
        DevicePool::get().tick();
    }
};

}  // namespace lvrhip
