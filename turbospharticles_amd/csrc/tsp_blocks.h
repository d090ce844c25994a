// tsp_blocks.h -- device memory of the contexts of a process: what each holds, and the released blocks
// that it keeps for its next layout.
//
// A scene pulled anew asks for mostly the same 83 blocks that the replaced layout releases; freeing and
// allocating them took 9.4 of the 11.7 ms of a pull at 1M particles (hipFree unmaps). So a context keeps
// released blocks, at most kMost bytes of them (an 8M scene replaces 2.4 GB: with 0.7 GB kept its frame takes
// 62 ms for 55) and kMostOnDevice over all contexts of a device (3% of it), and they are given back when
// any context of the process runs out of memory on that device, on trim, and with the context. Other
// users of the device do not reach them: tsp_trim is for those.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <map>
#include <mutex>

namespace tsp
{
    class Blocks
    {
    public:
        static constexpr uint64_t kMost = 2ull << 30;
        static constexpr uint64_t kMostOnDevice = 8ull << 30;

        Blocks() = default;
        Blocks(const Blocks&) = delete;
        Blocks& operator=(const Blocks&) = delete;
        ~Blocks()
        {
            trim();
            std::lock_guard<std::mutex> lock(mutex());
            for (Blocks** at = &first(); *at; at = &(*at)->next) { if (*at == this) { *at = next; break; } }
        }

        // the device of the context (once, before the first block)
        void join(int device)
        {
            dev = device;
            std::lock_guard<std::mutex> lock(mutex());
            next = first();
            first() = this;
        }

        // the most bytes that all contexts of the device may hold when this one allocates
        void setLimit(uint64_t bytes)
        {
            std::lock_guard<std::mutex> lock(mutex());
            limit = bytes;
        }

        // a block of at least `bytes` (its size comes back): a kept one that is not much larger, or new
        // memory, for which the device's kept blocks are given back when it has no other
        hipError_t take(uint64_t bytes, void** p, uint64_t* size)
        {
            std::lock_guard<std::mutex> lock(mutex());
            const auto it = kept.lower_bound(bytes);
            if (it != kept.end() && it->first <= bytes + bytes / 8u + 256u)
            {
                *size = it->first;
                *p = it->second;
                keptBytes -= *size;
                kept.erase(it);
            }
            else
            {
                *size = bytes;
                hipError_t e = allocate(bytes, p);
                if (e == hipErrorOutOfMemory && dropAll()) { e = allocate(bytes, p); }
                if (e != hipSuccess) { return e; }
            }
            liveBytes += *size;
            peakBytes = std::max(peakBytes, liveBytes + keptBytes);
            return hipSuccess;
        }

        // a block that is no longer used (by work that precedes its next use on the context's streams)
        void release(void* p, uint64_t size) noexcept
        {
            if (!keep(p, size)) { (void)hipFree(p); }   // (outside the lock: it waits for the device)
        }

        // gives back what this context keeps
        void trim()
        {
            std::lock_guard<std::mutex> lock(mutex());
            drop();
        }

        // gives back what the contexts of the device keep; false when they kept nothing
        bool trimDevice()
        {
            std::lock_guard<std::mutex> lock(mutex());
            return dropAll();
        }

        // bytes kept, and held (in use and kept) now and at most
        void bytes(uint64_t* keptNow, uint64_t* held, uint64_t* peak) const
        {
            std::lock_guard<std::mutex> lock(mutex());
            *keptNow = keptBytes;
            *held = liveBytes + keptBytes;
            *peak = peakBytes;
        }

    private:
        // one lock and one list for the process; never destroyed, since contexts may outlive static objects
        static std::mutex& mutex()
        {
            static std::mutex* m = new std::mutex;
            return *m;
        }
        static Blocks*& first()
        {
            static Blocks* b = nullptr;
            return b;
        }

        hipError_t allocate(uint64_t bytes, void** p)
        {
            uint64_t held = bytes;
            for (const Blocks* b = first(); b; b = b->next) { if (b->dev == dev) { held += b->liveBytes + b->keptBytes; } }
            if (held > limit) { return hipErrorOutOfMemory; }
            const hipError_t e = hipMalloc(p, bytes);
            if (e != hipSuccess) { (void)hipGetLastError(); }
            return e;
        }

        bool keep(void* p, uint64_t size) noexcept
        {
            std::lock_guard<std::mutex> lock(mutex());
            liveBytes -= size;
            uint64_t all = size;
            for (const Blocks* b = first(); b; b = b->next) { if (b->dev == dev) { all += b->keptBytes; } }
            if (keptBytes + size > kMost || all > kMostOnDevice) { return false; }
            try
            {
                kept.emplace(size, p);
            }
            catch (...)
            {
                return false;   // no host memory for the record
            }
            keptBytes += size;
            return true;
        }

        // (hipFree waits for the work that uses the block)
        bool drop()
        {
            const bool any = !kept.empty();
            for (const auto& b : kept) { (void)hipFree(b.second); }
            kept.clear();
            keptBytes = 0;
            return any;
        }

        bool dropAll()
        {
            bool any = false;
            for (Blocks* b = first(); b; b = b->next) { if (b->dev == dev) { any = b->drop() || any; } }
            return any;
        }

        std::multimap<uint64_t, void*> kept;   // by size
        uint64_t keptBytes = 0, liveBytes = 0, peakBytes = 0;
        uint64_t limit = ~0ull;
        int dev = -1;
        Blocks* next = nullptr;
    };
}
