// kernels_transfer.hip -- fields of the state between the device records and the host.
//
// The host sees structure-of-arrays fields (tsp_state_view), the device holds packed records. The
// kernels here gather a batch of fields straight into pinned host memory, or scatter them from it, so
// that the host only copies contiguous ranges (from several threads when they are large) and a whole
// small scene takes one launch. Bound by the link (a kernel moves 8 MiB in 150 us, 56 GB/s) and by the
// page faults of the caller's new arrays. Against packing and unpacking on one host thread around
// pageable copies, 1M fluid particles: pulled in 2.8 to 3.6 ms for 19 to 28 (with the kept blocks of
// tsp_ctx::alloc), pushed in 5.6 for 26 to 33; 64k: 0.8 for 1.4 and 0.7 to 1.1 for 1.4.
#include "tsp_device.h"
#include "tsp_transfer.h"

namespace tsp
{
    // one block per kXferBlock words of a piece
    template <bool kOut>
    __global__ void __launch_bounds__(kBlock) kTransfer(XferBatch b, uint32_t* __restrict__ stage)
    {
        uint32_t q = 0;
        while (q + 1u < b.count && blockIdx.x >= b.block[q + 1u]) { q++; }
        const XferPiece& p = b.piece[q];
        const uint32_t i0 = (blockIdx.x - b.block[q]) * kXferBlock + threadIdx.x;
        constexpr uint32_t kEach = kXferBlock / kBlock;
        uint32_t* w[kEach];
        uint32_t v[kEach];
#pragma unroll
        for (uint32_t u = 0; u < kEach; u++)
        {
            const uint32_t i = i0 + u * kBlock;
            const uint32_t word = p.first + (i < p.n ? i : 0u);
            const uint32_t rec = p.comps == 1u ? word : word / p.comps;
            w[u] = reinterpret_cast<uint32_t*>(p.dev + static_cast<size_t>(rec) * p.stride) + (word - rec * p.comps);
            v[u] = kOut ? *w[u] : stage[p.at + (i < p.n ? i : 0u)];
        }
#pragma unroll
        for (uint32_t u = 0; u < kEach; u++)
        {
            const uint32_t i = i0 + u * kBlock;
            if (i >= p.n) { continue; }
            if (kOut) { stage[p.at + i] = v[u]; } else { *w[u] = v[u]; }
        }
    }

    void launchTransfer(hipStream_t s, bool out, const XferBatch& b, uint32_t* stage)
    {
        const uint32_t n = b.block[b.count];
        if (!n) { return; }
        if (out) { kTransfer<true><<<n, kBlock, 0, s>>>(b, stage); }
        else { kTransfer<false><<<n, kBlock, 0, s>>>(b, stage); }
    }

    // sort keys as a caller sees them: scene-local Morton ids in 64 bits, all ones outside the frame
    __global__ void __launch_bounds__(kBlock) kLocalKeys(Dev d, const uint32_t* __restrict__ key, uint32_t off, uint32_t n,
                                                         uint64_t base, uint64_t empty, uint64_t* __restrict__ out)
    {
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i >= n) { return; }
        const uint64_t k = keyAt(d, key, off + i);
        out[i] = k >= empty ? ~0ull : k - base;
    }

    // order relative to the scene's first slot
    __global__ void __launch_bounds__(kBlock) kLocalOrder(const uint32_t* __restrict__ idx, uint32_t off, uint32_t n,
                                                          uint32_t* __restrict__ out)
    {
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i < n) { out[i] = idx[off + i] - off; }
    }

    static inline uint32_t blocksN(uint64_t n) { return static_cast<uint32_t>((n + kBlock - 1) / kBlock); }

    void launchLocalKeys(hipStream_t s, const Dev& d, const uint32_t* key, uint32_t off, uint32_t n, uint64_t base, uint64_t empty,
                         uint64_t* out)
    {
        if (n) { kLocalKeys<<<blocksN(n), kBlock, 0, s>>>(d, key, off, n, base, empty, out); }
    }

    void launchLocalOrder(hipStream_t s, const uint32_t* idx, uint32_t off, uint32_t n, uint32_t* out)
    {
        if (n) { kLocalOrder<<<blocksN(n), kBlock, 0, s>>>(idx, off, n, out); }
    }
}
