// tsp_transfer.h -- pieces of state fields that one launch moves between device records and pinned
// host memory (kernels_transfer.hip), and the host's copies between that memory and the caller's.
#pragma once

#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <thread>
#include <vector>

namespace tsp
{
    // n words of a field from its word `first` on, at stage[at ...]: word w is component w % comps of
    // the record at dev + (w / comps) * stride
    struct XferPiece
    {
        char* dev;
        uint32_t stride, comps, first, n, at, pad;
    };

    constexpr uint32_t kXferPieces = 64;     // pieces of a launch (the batch is a kernel argument)
    constexpr uint32_t kXferBlock = 1024;    // words per thread block

    struct XferBatch
    {
        XferPiece piece[kXferPieces];
        uint32_t block[kXferPieces + 1];     // first thread block of each piece; block[count] their number
        uint32_t count;
    };

    // a field of the caller and its device records, in 4-byte words: n of them, comps to a record
    struct XferField
    {
        char* host;
        char* dev;
        uint32_t stride, comps;
        uint64_t n;
    };

    // words [done, done + n) of a field, at stage[at ...]. The piece starts at the record of its first word,
    // so that its word numbers stay small however long the field is (three words each of 2^31 records pass 2^32).
    inline XferPiece pieceOf(const XferField& f, uint64_t done, uint32_t n, uint32_t at)
    {
        const uint64_t rec = done / f.comps;
        return XferPiece{ f.dev + rec * f.stride, f.stride, f.comps, static_cast<uint32_t>(done - rec * f.comps), n, at, 0u };
    }

    // a range of the stage and where it belongs in the caller's memory
    struct StageCopy
    {
        char* host;
        size_t at, bytes;
    };

    // the copies of one stage, by several threads when they are worth it: a thread moves about 8 GB/s
    // (less where it faults in new pages), the link 57
    inline void copyStage(const std::vector<StageCopy>& copies, char* stage, bool out)
    {
        constexpr size_t kPerThread = 512u << 10;
        constexpr size_t kMaxThreads = 8;
        size_t total = 0;
        for (const StageCopy& c : copies) { total += c.bytes; }
        const size_t threads = std::max<size_t>(1, std::min(kMaxThreads, total / kPerThread));
        const auto work = [&](size_t t)
        {
            // bytes [lo, hi) of the copies laid end to end
            const size_t lo = total * t / threads, hi = total * (t + 1) / threads;
            size_t pos = 0;
            for (const StageCopy& c : copies)
            {
                const size_t a = std::max(lo, pos), b = std::min(hi, pos + c.bytes);
                if (a < b)
                {
                    char* h = c.host + (a - pos);
                    char* s = stage + c.at + (a - pos);
                    if (out) { memcpy(h, s, b - a); } else { memcpy(s, h, b - a); }
                }
                pos += c.bytes;
            }
        };
        std::vector<std::thread> pool;
        size_t started = 1;
        try
        {
            pool.reserve(threads);
            for (; started < threads; started++) { pool.emplace_back(work, started); }
        }
        catch (...)
        {
            // no thread to be had: the rest is copied here
        }
        work(0);
        for (size_t t = started; t < threads; t++) { work(t); }
        for (std::thread& t : pool) { t.join(); }
    }
}
