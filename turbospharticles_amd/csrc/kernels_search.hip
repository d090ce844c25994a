// kernels_search.hip -- neighbor search of the IISPH step on gfx950.
//
// Re-order (DataReOrder_SolverStep), Construct and Query of the reference's compact
// cell-linked list, written for wave64:
//   keys      Morton cell id of every particle in the local cell frame, with the frame
//             hysteresis test of UpdateCellFrame (CPU/backend/neighbor_search.cpp:1902-1960)
//   sort      stable LSD radix sort of (key, index), 8-bit digits, keys clamped so that
//             out-of-frame particles sort last (neighbor_search.cpp:403-564); per tile the
//             stable ranks come from wave64 ballots, not from a serial scan
//   permute   one gather of the packed particle records per particle
//   cells     dense {begin, end} table over the frame, written at the runs of the sorted keys;
//             the previous step's runs are cleared first, so no global counter is needed
//   count     per particle: FF/FB/FR hit masks and counts over the 27-cell stencil (inclusive
//             cutoff, distance fma(dx,dx,fma(dy,dy,dz*dz)), neighbor_search.cpp:1130-1249); per
//             64-position slice: pitch, base, u16/u32 format and storage
//   scan      one-pass exclusive scans of many blocks (RF, RB and RR offsets, the surface flags of an export)
//   fill      writes the entries in the reference's iteration order: z-y-x stencil raster,
//             ascending index within a cell (CPU/backend/neighbor_lists.h:171-197 for wide lists),
//             and builds the FF halo of each 256-particle block
#include "tsp_device.h"

namespace tsp
{
    // ----------------------------------------------------------------------------------------
    // multi-block exclusive scan of u32 values (tiles of 2048 = 256 threads x 8)

    constexpr uint32_t kScanTile = 2048;

    // exclusive scan over the lanes of a wave; sum: the wave's total in every lane
    __device__ __forceinline__ uint32_t waveExclusiveScan(uint32_t v, uint32_t& sum)
    {
        const uint32_t lane = threadIdx.x & 63u;
        uint32_t incl = v;
        for (int o = 1; o < 64; o <<= 1)
        {
            const uint32_t u = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), o, 64));
            if (lane >= static_cast<uint32_t>(o)) { incl += u; }
        }
        sum = static_cast<uint32_t>(__shfl(static_cast<int>(incl), 63, 64));
        return incl - v;
    }

    // exclusive scan over the first kBlock threads of a block (the others pass and get anything)
    __device__ __forceinline__ uint32_t blockExclusiveScan(uint32_t v, uint32_t& total)
    {
        __shared__ uint32_t tot[kBlock / 64];
        uint32_t sum;
        uint32_t r = waveExclusiveScan(v, sum);
        const uint32_t wave = threadIdx.x >> 6;
        if (wave < kBlock / 64 && (threadIdx.x & 63u) == 0u) { tot[wave] = sum; }
        __syncthreads();
        total = 0;
        for (uint32_t w = 0; w < kBlock / 64; w++)
        {
            if (w < wave) { r += tot[w]; }
            total += tot[w];
        }
        return r;
    }

    // Decoupled look-back (Merrill & Garland 2016), for the scan and the sort passes: each block takes
    // the next tile number from a counter, so a tile waits only on tiles whose blocks started before
    // it; it publishes its sum, adds its predecessors' sums walking back to the first inclusive
    // prefix, publishes that prefix and writes its values. Status words carry the launch's epoch
    // (bit 33 up), a prefix flag (bit 32) and the value in one 64-bit word, so the polls need no
    // ordering and no clearing pass is needed: the last block resets the counter and counts the
    // launch in the epoch word. A launch's epoch is 1 + (launches before it mod 2^31 - 1), never 0,
    // so the zeroed state of a new buffer matches no launch. A wait longer than kScanSpins polls
    // gives up and sets the fail word (never expected; the host reports it).
    // A walk reads many predecessors at a time: a poll is a round trip to memory (the XCDs share no
    // L2).
    constexpr uint32_t kScanSpins = 1u << 20;
    constexpr unsigned long long kScanPrefix = 1ull << 32;

    __device__ __forceinline__ unsigned long long scanTag(uint32_t epoch)
    {
        return static_cast<unsigned long long>(epoch % 0x7fffffffu + 1u) << 33;
    }

    __device__ __forceinline__ unsigned long long pollStatus(const unsigned long long* w)
    {
        return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    __device__ __forceinline__ void publishStatus(unsigned long long* w, unsigned long long v)
    {
        __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // the sum of the tiles before `tile` (> 0), by one whole wave: 64 predecessors at a time
    __device__ __forceinline__ uint32_t lookBackWave(const unsigned long long* status, uint32_t tile, unsigned long long tag,
        uint32_t* fail)
    {
        const uint32_t lane = threadIdx.x & 63u;
        uint32_t prefix = 0, spins = 0;
        uint32_t left = tile;   // tiles not added yet: 0 .. left - 1
        for (;;)
        {
            const unsigned long long w = lane < left ? pollStatus(&status[left - 1u - lane]) : 0ull;
            const bool ready = (w >> 33) == (tag >> 33);
            const uint64_t readyMask = __ballot(ready);
            const uint64_t prefMask = __ballot(ready && (w & kScanPrefix) != 0ull);
            // lanes of the unbroken run of ready tiles, up to the first prefix
            uint32_t run = readyMask == ~0ull ? 64u : static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(~readyMask))) - 1u;
            const uint32_t pre = prefMask == 0ull ? 64u : static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(prefMask))) - 1u;
            const bool done = pre < run;
            if (done) { run = pre + 1u; }
            uint32_t v = lane < run ? static_cast<uint32_t>(w) : 0u;
            for (int o = 32; o > 0; o >>= 1) { v += static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), o, 64)); }
            prefix += v;
            left -= run;
            if (done || left == 0u) { return prefix; }
            if (run == 0u)
            {
                if (++spins > kScanSpins)
                {
                    if (lane == 0u) { atomicOr(fail, 1u); }
                    return prefix;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
    }

    // One-pass exclusive scan. 8 M values (3,907 tiles): 178 us, 2,070 with one thread walking back tile by tile.
    __global__ void __launch_bounds__(kBlock) kScanOnePass(uint32_t* __restrict__ v, uint32_t m, uint32_t* __restrict__ tmp,
        uint32_t* __restrict__ fail)
    {
        __shared__ uint32_t sTile, sEpoch, sPrefix;
        uint32_t* counter = tmp;
        uint32_t* epochWord = tmp + 1;
        unsigned long long* status = reinterpret_cast<unsigned long long*>(tmp + kScanHeaderWords);
        const uint32_t nb = (m + kScanTile - 1) / kScanTile;
        if (threadIdx.x == 0)
        {
            sEpoch = __hip_atomic_load(epochWord, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sTile = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        const uint32_t tile = sTile;
        const unsigned long long tag = scanTag(sEpoch);
        const uint32_t base = tile * kScanTile + threadIdx.x * 8u;
        uint32_t loc[8];
        uint32_t sum = 0;
        for (uint32_t q = 0; q < 8; q++) { loc[q] = base + q < m ? v[base + q] : 0u; sum += loc[q]; }
        uint32_t total;
        const uint32_t r = blockExclusiveScan(sum, total);
        if (threadIdx.x < 64u)
        {
            uint32_t prefix = 0;
            if (tile > 0)
            {
                if (threadIdx.x == 0) { publishStatus(&status[tile], tag | total); }
                prefix = lookBackWave(status, tile, tag, fail);
            }
            if (threadIdx.x == 0)
            {
                publishStatus(&status[tile], tag | kScanPrefix | (prefix + total));
                sPrefix = prefix;
                if (tile == nb - 1)
                {
                    // every block has drawn its tile: ready the counter and epoch for the next scan
                    __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(epochWord, sEpoch + 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        }
        __syncthreads();
        uint32_t run = sPrefix + r;
        for (uint32_t q = 0; q < 8; q++)
        {
            if (base + q < m) { v[base + q] = run; }
            run += loc[q];
        }
    }

    // exclusive scan of m values in place; tmp is a scan state of scanTmpWords(m) words, zeroed
    // when allocated (fail: set if a look-back gave up)
    void launchScan(hipStream_t s, uint32_t* v, uint32_t m, uint32_t* tmp, uint32_t* fail)
    {
        if (m == 0) { return; }
        const uint32_t nb = (m + kScanTile - 1) / kScanTile;
        kScanOnePass<<<nb, kBlock, 0, s>>>(v, m, tmp, fail);
    }

    // ----------------------------------------------------------------------------------------
    // keys

    __device__ __forceinline__ bool insideDomain(const Frame& f, float x, float y, float z)
    {
        if (!f.domainSet) { return true; }
        return x >= f.domMin[0] && x <= f.domMax[0] && y >= f.domMin[1] && y <= f.domMax[1]
            && z >= f.domMin[2] && z <= f.domMax[2];
    }

    // cell id of one position in its scene's key range; sets the abort flags when an in-domain
    // particle left the inner frame
    __device__ __forceinline__ uint64_t cellKey(const Frame& f, float x, float y, float z, bool check, Status* st, Solve* so)
    {
        const int cx = floorToInt(x * f.cellSizeInv);
        const int cy = floorToInt(y * f.cellSizeInv);
        const int cz = floorToInt(z * f.cellSizeInv);
        if (check && insideDomain(f, x, y, z))
        {
            if (cx < f.innerLo[0] || cx > f.innerHi[0] || cy < f.innerLo[1] || cy > f.innerHi[1]
                || cz < f.innerLo[2] || cz > f.innerHi[2])
            {
                atomicOr(&st->abort, 1u);
                atomicOr(&so->abort, 1u);
            }
        }
        const int lx = cx - f.orig[0], ly = cy - f.orig[1], lz = cz - f.orig[2];
        if (lx < 0 || lx >= static_cast<int>(f.dim[0]) || ly < 0 || ly >= static_cast<int>(f.dim[1])
            || lz < 0 || lz >= static_cast<int>(f.dim[2]))
        {
            return f.emptyKey;
        }
        return f.keyBase + morton64(static_cast<uint32_t>(lx), static_cast<uint32_t>(ly), static_cast<uint32_t>(lz));
    }

    enum Pop { POP_F = 0, POP_B = 1, POP_R = 2 };

    __device__ __forceinline__ uint32_t sceneOfParticle(const Dev& d, int pop, uint32_t i)
    {
        if (pop == POP_F) { return d.blockScene[i / kBlock]; }
        if (pop == POP_B) { return d.sceneB[i]; }
        return d.bodyScene[d.rbody[i]];
    }

    // key of particle i of a population; the padding slots of a fluid segment take the dead key
    __device__ __forceinline__ uint64_t particleKey(const Dev& d, int pop, const float4* p, uint32_t i, bool check)
    {
        const uint32_t s = sceneOfParticle(d, pop, i);
        const Frame& f = d.frames[s];
        if (pop == POP_F && i - d.scenes[s].offF >= d.scenes[s].nF) { return f.deadKey; }
        const float4 q = p[i];
        return cellKey(f, q.x, q.y, q.z, check, d.status, &d.solve[s]);
    }

    // the digits of a key counted in LDS, cnt[pass][digit]
    template <typename K>
    __device__ __forceinline__ void countDigits(uint32_t (&cnt)[kRadixPasses<K>][kRadixBins], K k, uint32_t passes)
    {
#pragma unroll
        for (uint32_t q = 0; q < kRadixPasses<K>; q++)
        {
            if (q < passes) { atomicAdd(&cnt[q][static_cast<uint32_t>(k >> (q * kRadixBits)) & (kRadixBins - 1u)], 1u); }
        }
    }

    template <typename K>
    __device__ __forceinline__ void clearDigits(uint32_t (&cnt)[kRadixPasses<K>][kRadixBins], uint32_t passes)
    {
        for (uint32_t q = 0; q < passes; q++) { cnt[q][threadIdx.x] = 0u; }
        __syncthreads();
    }

    template <typename K>
    __device__ __forceinline__ void addDigits(const uint32_t (&cnt)[kRadixPasses<K>][kRadixBins], uint32_t passes,
        uint32_t* __restrict__ state)
    {
        __syncthreads();
        for (uint32_t q = 0; q < passes; q++)
        {
            const uint32_t c = cnt[q][threadIdx.x];
            if (c) { atomicAdd(&state[kRadixHeaderWords + q * kRadixBins + threadIdx.x], c); }
        }
    }

    // keys and indices of a population; passes > 0 adds the digit counts of all sort passes to the sort
    // state (particles in motion are nearly in order, so a block meets few digits and adds few words)
    template <typename K>
    __global__ void __launch_bounds__(kBlock) kKeys(Dev d, int pop, const float4* __restrict__ p, uint32_t n, bool check,
        K* __restrict__ key, uint32_t* __restrict__ idx, uint32_t* __restrict__ state, uint32_t passes)
    {
        __shared__ uint32_t cnt[kRadixPasses<K>][kRadixBins];
        if (passes) { clearDigits<K>(cnt, passes); }
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i < n)
        {
            const K k = static_cast<K>(particleKey(d, pop, p, i, check));
            key[i] = k;
            idx[i] = i;
            countDigits<K>(cnt, k, passes);
        }
        if (passes) { addDigits<K>(cnt, passes, state); }
    }

    // the digit counts of keys that another kernel wrote
    template <typename K>
    __global__ void __launch_bounds__(kBlock) kRadixCount(const K* __restrict__ key, uint32_t n, uint32_t* __restrict__ state,
        uint32_t passes)
    {
        __shared__ uint32_t cnt[kRadixPasses<K>][kRadixBins];
        clearDigits<K>(cnt, passes);
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i < n) { countDigits<K>(cnt, key[i], passes); }
        addDigits<K>(cnt, passes, state);
    }

    // boundary keys; flags a descent so the host knows whether the order needs a sort
    template <typename K>
    __global__ void __launch_bounds__(kBlock) kKeysSorted(Dev d, const float4* __restrict__ p, uint32_t n,
        K* __restrict__ key, uint32_t* __restrict__ idx)
    {
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i >= n) { return; }
        const uint64_t k = particleKey(d, POP_B, p, i, false);
        key[i] = static_cast<K>(k);
        idx[i] = i;
        if (i > 0 && particleKey(d, POP_B, p, i - 1, false) > k) { atomicOr(&d.status->bUnsorted, 1u); }
    }

    // ----------------------------------------------------------------------------------------
    // stable LSD radix sort, 8-bit digits, in three forms by the number of keys.
    //   up to 2^14   one launch of one block (kSortSmall)
    //   up to 2^18   one launch per digit (kRadixPass): the counts of all digits come first, with the keys
    //                (they do not depend on the order); a tile ranks its keys, publishes its digit counts,
    //                adds up those of the tiles before it by decoupled look-back (one digit per thread)
    //                and writes its keys
    //   more         three launches per digit (kRadixHist, kRadixDigitScan, kRadixScatter)
    // Look-back saves six of ten launches, which is most of a small sort's time (64,000 particles: 66 us of
    // kernels in ten launches to 39 us in four), but every poll passes the L2s by: with 489 tiles a pass
    // took 48 us, with 3,907 tiles 333 to 505, against 19 and 75 to 100 in three launches. With the scan
    // of all counts by one look-back between them, in place of one block per digit, those three took 34 and 242.

    // ranks of one wave's keys among those of the same digit, in key order (round r, then lane);
    // cnt: the wave's digit counts, zeroed before and complete after. The counter is read by all lanes
    // of a digit and then advanced by the lowest one: LDS serves a wave's accesses in order, the fences
    // keep the compiler to it.
    template <typename K, uint32_t kPer>
    __device__ __forceinline__ void rankWave(uint32_t* cnt, const K (&k)[kPer], uint32_t first, uint32_t n, uint32_t shift,
        uint32_t bits, uint32_t (&rank)[kPer])
    {
        const uint32_t digitBits = min(kRadixBits, bits - shift);   // the key's bits end here
        const uint32_t lane = threadIdx.x & 63u;
        const uint64_t lanesBelow = (lane == 0) ? 0ull : (~0ull >> (64u - lane));
#pragma unroll
        for (uint32_t r = 0; r < kPer; r++)
        {
            rank[r] = 0u;
            if (first + r * 64u >= n) { continue; }
            const bool valid = first + r * 64u + lane < n;
            const uint32_t dg = static_cast<uint32_t>(k[r] >> shift) & (kRadixBins - 1u);
            uint64_t match = __ballot(valid);
#pragma unroll
            for (uint32_t bit = 0; bit < kRadixBits; bit++)
            {
                if (bit >= digitBits) { break; }
                const bool set = (dg >> bit) & 1u;
                const uint64_t bs = __ballot(set);
                match &= set ? bs : ~bs;
            }
            const uint32_t below = __popcll(match & lanesBelow);
            if (valid)
            {
                const uint32_t before = cnt[dg];
                rank[r] = before + below;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                if (below == 0u) { cnt[dg] = before + __popcll(match); }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }

    // the sum of one digit's counts in the tiles before `tile` (> 0), by one thread per digit: eight
    // predecessors at a time
    __device__ __forceinline__ uint32_t lookBackDigit(const unsigned long long* status, uint32_t tile, uint32_t digit,
        unsigned long long tag, uint32_t* fail)
    {
        constexpr uint32_t kAhead = 8;
        uint32_t prefix = 0, spins = 0;
        uint32_t left = tile;
        for (;;)
        {
            unsigned long long w[kAhead];
#pragma unroll
            for (uint32_t q = 0; q < kAhead; q++)
            {
                w[q] = q < left ? pollStatus(&status[static_cast<uint64_t>(left - 1u - q) * kRadixBins + digit]) : 0ull;
            }
            uint32_t run = 0;
            bool open = true, done = false;
#pragma unroll
            for (uint32_t q = 0; q < kAhead; q++)
            {
                open = open && !done && (w[q] >> 33) == (tag >> 33);
                if (open)
                {
                    prefix += static_cast<uint32_t>(w[q]);
                    run++;
                    done = (w[q] & kScanPrefix) != 0ull;
                }
            }
            left -= run;
            if (done || left == 0u) { return prefix; }
            if (run == 0u)
            {
                if (++spins > kScanSpins)
                {
                    atomicOr(fail, 1u);
                    return prefix;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
    }

    // what a sort pass's two forms share: a tile's keys in registers, ranked wave by wave; then, with the
    // place of the tile's first key of digit t known to thread t, every key's place
    template <typename K, uint32_t kPer>
    struct TileKeys
    {
        static constexpr uint32_t kWaves = kBlock / 64;
        K k[kPer];
        uint32_t ix[kPer], rank[kPer], c[kWaves];
        uint32_t first;

        // cnt: zeroed; the tile's count of digit t comes back in thread t
        __device__ __forceinline__ uint32_t load(uint32_t (&cnt)[kWaves][kRadixBins], const K* __restrict__ keyIn,
            const uint32_t* __restrict__ idxIn, uint32_t tile, uint32_t n, uint32_t shift, uint32_t bits)
        {
            const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
            first = tile * (kBlock * kPer) + wave * (64u * kPer);
#pragma unroll
            for (uint32_t r = 0; r < kPer; r++)
            {
                const uint32_t i = first + r * 64u + lane;
                k[r] = i < n ? keyIn[i] : K(0);
                ix[r] = i < n ? idxIn[i] : 0u;
            }
            rankWave<K, kPer>(cnt[wave], k, first, n, shift, bits, rank);
            __syncthreads();
            uint32_t total = 0;
            for (uint32_t w = 0; w < kWaves; w++) { c[w] = cnt[w][threadIdx.x]; total += c[w]; }
            return total;
        }

        __device__ __forceinline__ void store(uint32_t (&cnt)[kWaves][kRadixBins], K* __restrict__ keyOut,
            uint32_t* __restrict__ idxOut, uint32_t at, uint32_t n, uint32_t shift)
        {
            const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
            for (uint32_t w = 0; w < kWaves; w++) { cnt[w][threadIdx.x] = at; at += c[w]; }
            __syncthreads();
#pragma unroll
            for (uint32_t r = 0; r < kPer; r++)
            {
                if (first + r * 64u + lane < n)
                {
                    const uint32_t o = cnt[wave][static_cast<uint32_t>(k[r] >> shift) & (kRadixBins - 1u)] + rank[r];
                    // (out of range only after a look-back gave up)
                    if (o < n) { keyOut[o] = k[r]; idxOut[o] = ix[r]; }
                }
            }
        }
    };

    // one digit of a sort with few tiles. state: the header (tile counter, epoch, blocks that have read),
    // the digit counts of all passes and the tiles' status words. The block that reads them last clears
    // what this pass used.
    template <typename K, uint32_t kPer>
    __global__ void __launch_bounds__(kBlock) kRadixPass(const K* __restrict__ keyIn, const uint32_t* __restrict__ idxIn,
        K* __restrict__ keyOut, uint32_t* __restrict__ idxOut, uint32_t n, uint32_t pass, uint32_t bits,
        uint32_t* __restrict__ state, uint32_t* __restrict__ fail)
    {
        constexpr uint32_t kWaves = kBlock / 64;
        static_assert(kRadixBins == kBlock, "one digit per thread");
        __shared__ uint32_t cnt[kWaves][kRadixBins];
        __shared__ uint32_t sHist[kRadixBins];
        __shared__ uint32_t sTile, sEpoch, sLast;
        uint32_t* hist = state + kRadixHeaderWords + pass * kRadixBins;
        unsigned long long* status = reinterpret_cast<unsigned long long*>(state + kRadixStatusAt);
        const uint32_t t = threadIdx.x;
        if (t == 0)
        {
            sEpoch = __hip_atomic_load(&state[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            sTile = __hip_atomic_fetch_add(&state[0], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        }
        sHist[t] = hist[t];
        for (uint32_t w = 0; w < kWaves; w++) { cnt[w][t] = 0u; }
        __syncthreads();
        // this block has what it reads of the state (the counts are in LDS); its turn among the blocks
        // comes back while the keys load, and is looked at when they are placed
        uint32_t readers = 0;
        if (t == 0) { readers = __hip_atomic_fetch_add(&state[2], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
        const uint32_t tile = sTile;
        const unsigned long long tag = scanTag(sEpoch);
        TileKeys<K, kPer> keys;
        const uint32_t total = keys.load(cnt, keyIn, idxIn, tile, n, pass * kRadixBits, bits);
        unsigned long long* mine = &status[static_cast<uint64_t>(tile) * kRadixBins + t];
        publishStatus(mine, tag | (tile == 0u ? kScanPrefix : 0ull) | total);
        uint32_t all;
        uint32_t at = blockExclusiveScan(sHist[t], all);
        if (tile > 0u)
        {
            const uint32_t prefix = lookBackDigit(status, tile, t, tag, fail);
            publishStatus(mine, tag | kScanPrefix | (prefix + total));
            at += prefix;
        }
        if (t == 0) { sLast = readers == gridDim.x - 1u; }
        keys.store(cnt, keyOut, idxOut, at, n, pass * kRadixBits);   // (a barrier after sLast is written)
        if (sLast)
        {
            hist[t] = 0u;
            if (t == 0)
            {
                __hip_atomic_store(&state[0], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&state[2], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(&state[1], sEpoch + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }

    // one digit of a sort with many tiles, in three launches: the tiles' digit counts (hist[digit][tile]),
    // their exclusive scan along the tiles of each digit (a block per digit: no block waits for another),
    // and the scatter, which adds the digits before.
    constexpr uint32_t kManyPer = kRadixManyTile / kBlock;

    template <typename K>
    __global__ void __launch_bounds__(kBlock) kRadixHist(const K* __restrict__ key, uint32_t n, uint32_t shift,
        uint32_t nTiles, uint32_t* __restrict__ hist)
    {
        __shared__ uint32_t cnt[kRadixBins];
        cnt[threadIdx.x] = 0;
        __syncthreads();
        const uint32_t base = blockIdx.x * kRadixManyTile + threadIdx.x;
#pragma unroll
        for (uint32_t r = 0; r < kManyPer; r++)
        {
            const uint32_t i = base + r * kBlock;
            if (i < n) { atomicAdd(&cnt[static_cast<uint32_t>(key[i] >> shift) & (kRadixBins - 1u)], 1u); }
        }
        __syncthreads();
        hist[threadIdx.x * nTiles + blockIdx.x] = cnt[threadIdx.x];
    }

    __global__ void __launch_bounds__(kBlock) kRadixDigitScan(uint32_t* __restrict__ hist, uint32_t nTiles,
        uint32_t* __restrict__ totals)
    {
        uint32_t* row = hist + static_cast<uint64_t>(blockIdx.x) * nTiles;
        uint32_t before = 0;
        for (uint32_t b = 0; b < nTiles; b += kRadixManyTile)
        {
            const uint32_t base = b + threadIdx.x * kManyPer;
            uint32_t loc[kManyPer], sum = 0;
#pragma unroll
            for (uint32_t q = 0; q < kManyPer; q++) { loc[q] = base + q < nTiles ? row[base + q] : 0u; sum += loc[q]; }
            uint32_t total;
            uint32_t run = before + blockExclusiveScan(sum, total);
            __syncthreads();
#pragma unroll
            for (uint32_t q = 0; q < kManyPer; q++)
            {
                if (base + q < nTiles) { row[base + q] = run; }
                run += loc[q];
            }
            before += total;
        }
        if (threadIdx.x == 0) { totals[blockIdx.x] = before; }
    }

    template <typename K>
    __global__ void __launch_bounds__(kBlock) kRadixScatter(const K* __restrict__ keyIn, const uint32_t* __restrict__ idxIn,
        K* __restrict__ keyOut, uint32_t* __restrict__ idxOut, uint32_t n, uint32_t shift, uint32_t bits, uint32_t nTiles,
        const uint32_t* __restrict__ hist, const uint32_t* __restrict__ totals)
    {
        __shared__ uint32_t cnt[kBlock / 64][kRadixBins];
        const uint32_t t = threadIdx.x;
        const uint32_t before = hist[t * nTiles + blockIdx.x];
        const uint32_t total = totals[t];
        for (uint32_t w = 0; w < kBlock / 64; w++) { cnt[w][t] = 0u; }
        __syncthreads();
        TileKeys<K, kManyPer> keys;
        keys.load(cnt, keyIn, idxIn, blockIdx.x, n, shift, bits);
        uint32_t all;
        const uint32_t at = blockExclusiveScan(total, all) + before;
        keys.store(cnt, keyOut, idxOut, at, n, shift);
    }

    // the whole sort of up to kSmallSort keys in one block of 1024 threads (one launch). A wave holds
    // 64 x kPer consecutive keys in registers and ranks them by itself; the 256 digits then add up the
    // waves' counts, and the keys and indices change places through LDS, a word at a time (64 KB for the
    // most keys, whatever their width).
    constexpr uint32_t kSmallThreads = 1024;
    constexpr uint32_t kSmallSort = kSmallThreads * 16;

    template <typename K, uint32_t kPer>
    __global__ void __launch_bounds__(kSmallThreads) kSortSmall(K* __restrict__ key, uint32_t* __restrict__ idx, uint32_t n,
        uint32_t bits)
    {
        constexpr uint32_t kWaves = kSmallThreads / 64;
        __shared__ uint32_t cnt[kWaves][kRadixBins];
        __shared__ uint32_t word[kSmallThreads * kPer];
        const uint32_t t = threadIdx.x;
        const uint32_t wave = t >> 6, lane = t & 63u;
        const uint32_t first = wave * (64u * kPer);
        K k[kPer];
        uint32_t ix[kPer], rank[kPer];
#pragma unroll
        for (uint32_t r = 0; r < kPer; r++)
        {
            const uint32_t i = first + r * 64u + lane;
            k[r] = i < n ? key[i] : K(0);
            ix[r] = i < n ? idx[i] : 0u;
        }
        const auto exchange = [&](auto&& get, auto&& set)
        {
#pragma unroll
            for (uint32_t r = 0; r < kPer; r++) { if (first + r * 64u + lane < n) { word[rank[r]] = get(r); } }
            __syncthreads();
#pragma unroll
            for (uint32_t r = 0; r < kPer; r++) { if (first + r * 64u + lane < n) { set(r, word[first + r * 64u + lane]); } }
            __syncthreads();
        };
        for (uint32_t shift = 0; shift < bits; shift += kRadixBits)
        {
            for (uint32_t w = t / kRadixBins; w < kWaves; w += kSmallThreads / kRadixBins) { cnt[w][t & (kRadixBins - 1u)] = 0u; }
            __syncthreads();
            rankWave<K, kPer>(cnt[wave], k, first, n, shift, bits, rank);
            __syncthreads();
            uint32_t c[kWaves];
            uint32_t total = 0;
            if (t < kRadixBins)
            {
#pragma unroll
                for (uint32_t w = 0; w < kWaves; w++) { c[w] = cnt[w][t]; total += c[w]; }
            }
            uint32_t all;
            uint32_t at = blockExclusiveScan(total, all);
            if (t < kRadixBins)
            {
#pragma unroll
                for (uint32_t w = 0; w < kWaves; w++) { cnt[w][t] = at; at += c[w]; }
            }
            __syncthreads();
#pragma unroll
            for (uint32_t r = 0; r < kPer; r++)
            {
                if (first + r * 64u + lane < n) { rank[r] += cnt[wave][static_cast<uint32_t>(k[r] >> shift) & (kRadixBins - 1u)]; }
            }
            // the digits of this pass are used up: the key itself moves, then its index
            if constexpr (sizeof(K) == 8)
            {
                exchange([&](uint32_t r) { return static_cast<uint32_t>(k[r] >> 32); },
                         [&](uint32_t r, uint32_t w) { k[r] = (static_cast<K>(w) << 32) | static_cast<uint32_t>(k[r]); });
            }
            exchange([&](uint32_t r) { return static_cast<uint32_t>(k[r]); },
                     [&](uint32_t r, uint32_t w) { k[r] = static_cast<K>((k[r] & ~static_cast<K>(0xffffffffu)) | w); });
            exchange([&](uint32_t r) { return ix[r]; }, [&](uint32_t r, uint32_t w) { ix[r] = w; });
        }
#pragma unroll
        for (uint32_t r = 0; r < kPer; r++)
        {
            const uint32_t i = first + r * 64u + lane;
            if (i < n) { key[i] = k[r]; idx[i] = ix[r]; }
        }
    }

    // ----------------------------------------------------------------------------------------
    // permutation (gather into the second buffers)

    __device__ __forceinline__ void gatherOne(const Gather& g, const uint32_t* __restrict__ idx, uint32_t i)
    {
        const uint32_t o = idx[i];
        for (uint32_t f = 0; f < g.n4; f++) { g.d4[f][i] = g.s4[f][o]; }
        for (uint32_t f = 0; f < g.n1; f++) { g.d1[f][i] = g.s1[f][o]; }
        if (g.idS) { g.idD[i] = g.idS[o]; }
    }

    __global__ void __launch_bounds__(kBlock) kPermute(Gather g, const uint32_t* __restrict__ idx)
    {
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i < g.n) { gatherOne(g, idx, i); }
    }

    // ----------------------------------------------------------------------------------------
    // cell tables

    // cell-table index of an in-frame key (local Morton id = key - keyBase)
    __device__ __forceinline__ uint32_t linearOfKey(const Frame& f, uint64_t k)
    {
        const uint64_t m = k - f.keyBase;
        return linearCell(f, compact21(m), compact21(m >> 1), compact21(m >> 2));
    }

    // the search status block and the scenes' frame-abort flags cleared, by one block
    __device__ __forceinline__ void resetSearch(const Dev& d)
    {
        constexpr uint32_t words = static_cast<uint32_t>(sizeof(Status) / sizeof(uint32_t));
        static_assert(words <= kBlock, "the reset covers one block");
        constexpr uint32_t keep = static_cast<uint32_t>(offsetof(Status, scanFail) / sizeof(uint32_t));
        if (threadIdx.x < words && threadIdx.x != keep) { reinterpret_cast<uint32_t*>(d.status)[threadIdx.x] = 0u; }
        for (uint32_t s = threadIdx.x; s < d.nScenes; s += kBlock)
        {
            Solve& so = d.solve[s];
            so.abort = 0u;
            so.contactActive = 0u; so.contactDone = 0u; so.contactIters = 0u; so.contactConverged = 0u;
            so.contactAvg = 0.0f; so.contactBoundary = 0u; so.contactBad = 0u; so.contacts = 0ull;
        }
    }

    // a search's start: the status block reset, and the cells of the runs of the previous sorted keys
    // (the only ones that are not empty) of the fluid and the rigid particles cleared
    __device__ __forceinline__ void clearCells(const Dev& d, const uint32_t* __restrict__ key, uint32_t i, uint32_t n,
        uint2* __restrict__ cell)
    {
        if (i >= n) { return; }
        const uint64_t k = keyAt(d, key, i);
        const Frame& f = d.frames[sceneOfKey(d, k)];
        if (k >= f.emptyKey) { return; }
        if (i == 0 || keyAt(d, key, i - 1) != k) { cell[linearOfKey(f, k)] = make_uint2(0u, 0u); }
    }

    __global__ void __launch_bounds__(kBlock) kResetSearch(Dev d, uint32_t blocksF)
    {
        if (blockIdx.x == 0u) { resetSearch(d); return; }
        const uint32_t b = blockIdx.x - 1u;
        if (b < blocksF) { clearCells(d, d.keyF, b * kBlock + threadIdx.x, d.nF, d.cellF); }
        else { clearCells(d, d.keyR, (b - blocksF) * kBlock + threadIdx.x, d.nR, d.cellR); }
    }

    __global__ void __launch_bounds__(kBlock) kClearAll(uint2* __restrict__ cell, uint64_t n)
    {
        const uint64_t q = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x;
        if (q < n) { cell[q] = make_uint2(0u, 0u); }
    }

    __device__ __forceinline__ void buildCells(const Dev& d, const uint32_t* __restrict__ key, uint32_t i, uint32_t n,
        uint2* __restrict__ cell)
    {
        const uint64_t k = keyAt(d, key, i);
        const Frame& f = d.frames[sceneOfKey(d, k)];
        if (k >= f.emptyKey) { return; }
        const bool first = i == 0 || keyAt(d, key, i - 1) != k;
        const bool last = i + 1 == n || keyAt(d, key, i + 1) != k;
        if (!first && !last) { return; }
        const uint32_t lin = linearOfKey(f, k);
        if (first) { cell[lin].x = i; }
        if (last) { cell[lin].y = i + 1; }
    }

    __global__ void __launch_bounds__(kBlock) kBuildCells(Dev d, const uint32_t* __restrict__ key, uint32_t n,
        uint2* __restrict__ cell)
    {
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i < n) { buildCells(d, key, i, n, cell); }
    }

    // the fluid's re-order and its cells
    __global__ void __launch_bounds__(kBlock) kPermuteCells(Dev d, Gather g)
    {
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i >= g.n) { return; }
        gatherOne(g, d.idxF, i);
        buildCells(d, d.keyF, i, g.n, d.cellF);
    }

    // ----------------------------------------------------------------------------------------
    // query: the 27-cell stencil in z-y-x raster order, one block of 768 threads per 256 particles.
    //
    // A wave takes 64 particles (one per lane) and three of the nine stencil rows (three x-adjacent
    // cells each), so three waves share a particle and a lane's chain of dependent candidate loads is a
    // third as long. The fill always runs so. The count pass does for up to kShareBlocks blocks (two per
    // CU: the chain is what its time consists of); beyond that one wave walks all nine rows, because
    // what the waves of a particle repeat, and their barriers, cost more than the shorter chain gains.
    // kQueryCount on a resting lattice, three waves / one wave: 16 blocks 30 / 49 us, 250 blocks 30 / 48, 311 blocks
    // 40 / 51, 432 blocks 42 / 50, 519 blocks 55 / 56, 686 blocks 60 / 56, 977 blocks 67 / 65, 2,000 blocks 111 /
    // 108, 3,907 blocks 202 / 179; against one lane walking all rows candidate by candidate: 16 blocks 66 to 33,
    // 432 blocks 82 to 49, 3,907 blocks 215 to 206, 31,250 blocks 1,333 to 1,205. What bounds the large launches is the vector
    // memory path: 240 scattered 12-byte records per lane, about 20 cycles a wave each. (Candidates
    // staged in LDS per 64 particles, in cell order: 250 us at 3,907 blocks, more barriers than loads
    // saved.)

    constexpr uint32_t kQueryThreads = 768;
    constexpr uint32_t kQueryShare = 3;          // waves per 64 particles
    static_assert(kQueryThreads == kBlock * kQueryShare, "three waves per 64 particles");
    constexpr uint32_t kShareBlocks = 512;       // most blocks that share particles in the count pass
    // the word after a particle's masks: rows whose fluid (boundary) candidates the masks do not cover;
    // all ones without masks
    constexpr uint32_t kOpenF = 0, kOpenB = kMaskRows;

    // the candidates of a stencil row: q -> q + (q < nA ? oA : oB). The cells 2m and 2m + 1 along x
    // have consecutive Morton keys, so three x-adjacent cells are two runs of the sorted particles,
    // ascending along the row.
    struct RowSpan
    {
        uint32_t nA, n, oA, oB;

        __device__ __forceinline__ uint32_t at(uint32_t q) const { return q + (q < nA ? oA : oB); }
    };

    // the row of the cells r[0..2], the first at an odd x or not
    __device__ __forceinline__ RowSpan rowSpan(const uint2 (&r)[3], bool odd)
    {
        const uint32_t n0 = r[0].y - r[0].x, n1 = r[1].y - r[1].x, n2 = r[2].y - r[2].x;
        RowSpan s;
        s.n = n0 + n1 + n2;
        s.nA = odd ? n0 : n0 + n1;
        s.oA = (odd || n0) ? r[0].x : r[1].x;
        s.oB = ((odd && n1) ? r[1].x : r[2].x) - s.nA;
        return s;
    }

    // the local cell of a particle, from its position as its key was made
    struct Cell
    {
        int l[3];
    };

    __device__ __forceinline__ Cell cellOf(const Frame& f, const float4& p)
    {
        return Cell{ { floorToInt(p.x * f.cellSizeInv) - f.orig[0], floorToInt(p.y * f.cellSizeInv) - f.orig[1],
                       floorToInt(p.z * f.cellSizeInv) - f.orig[2] } };
    }

    // the three cells of a row of the stencil, as loaded
    struct RowCells
    {
        uint2 r[3];
        bool odd;

        __device__ __forceinline__ RowSpan span() const { return rowSpan(r, odd); }
    };

    // The stencil of one particle: rows of side x side (y, z), each in chunks of three cells. Where the
    // stencils of the wave's active particles all lie inside a reach-1 frame (`near`: nearly always) a
    // row is one address; otherwise its cells are clamped to the frame. The loops over rows stay rolled:
    // a scene of few blocks pays for every instruction fetched, not only for those executed.
    struct Stencil
    {
        Cell at;
        uint32_t off, dx, dxy;   // first cell of the scene's tables, cells per y step, per z step
        uint32_t dim[3];
        int reach;
        uint32_t side, chunks;
        uint32_t first, last;    // the wave's rows
        bool near;

        // (lanes without `need` read the first cells of the tables and get an empty row)
        __device__ __forceinline__ RowCells cells(const uint2* __restrict__ table, uint32_t row, bool need) const
        {
            RowCells c;
            if (near)
            {
                const uint32_t zy = row;   // 3 (dz + 1) + dy + 1
                const uint32_t y = static_cast<uint32_t>(at.l[1]) + zy % 3u - 1u, z = static_cast<uint32_t>(at.l[2]) + zy / 3u - 1u;
                const uint32_t i = need ? off + static_cast<uint32_t>(at.l[0]) - 1u + dx * y + dxy * z : 0u;
#pragma unroll
                for (uint32_t q = 0; q < 3u; q++) { c.r[q] = table[i + q]; }
                if (!need) { for (uint32_t q = 0; q < 3u; q++) { c.r[q] = make_uint2(0u, 0u); } }
                c.odd = (at.l[0] & 1) == 0;
                return c;
            }
            const uint32_t k = row % chunks, zy = row / chunks;
            const int y = at.l[1] + static_cast<int>(zy % side) - reach, z = at.l[2] + static_cast<int>(zy / side) - reach;
            const int x0 = at.l[0] - reach + 3 * static_cast<int>(k), x = max(x0, 0);
            int nx = min(min(x0 + 2, at.l[0] + reach), static_cast<int>(dim[0]) - 1) - x + 1;
            if (!need || y < 0 || y >= static_cast<int>(dim[1]) || z < 0 || z >= static_cast<int>(dim[2])) { nx = 0; }
            const uint32_t i = off + static_cast<uint32_t>(x) + dx * static_cast<uint32_t>(y) + dxy * static_cast<uint32_t>(z);
#pragma unroll
            for (int q = 0; q < 3; q++) { c.r[q] = q < nx ? table[i + static_cast<uint32_t>(q)] : make_uint2(0u, 0u); }
            c.odd = (x & 1) != 0;
            return c;
        }
    };

    // share: which of the kShare waves of the 64 particles; active: the lane's particle is in the frame
    template <uint32_t kShare>
    __device__ __forceinline__ Stencil stencilOf(const Frame& f, const float4& p, bool active, uint32_t share)
    {
        Stencil s;
        s.at = cellOf(f, p);
        s.off = f.cellOff;
        s.dx = f.dim[0];
        s.dxy = f.dim[0] * f.dim[1];
        s.reach = f.reach;
        s.side = 2u * static_cast<uint32_t>(f.reach) + 1u;
        s.chunks = (s.side + 2u) / 3u;
        bool edge = false;
        for (int a = 0; a < 3; a++)
        {
            s.dim[a] = f.dim[a];
            edge = edge || s.at.l[a] < 1 || s.at.l[a] + 2 > static_cast<int>(f.dim[a]);
        }
        s.near = f.reach == 1 && !__any(active && edge);
        const uint32_t rows = s.side * s.side * s.chunks;
        s.first = rows * share / kShare;
        s.last = rows * (share + 1u) / kShare;
        return s;
    }

    __device__ __forceinline__ bool within(float xi, float yi, float zi, const float4& pj, float r2)
    {
        return dist2(xi - pj.x, yi - pj.y, zi - pj.z) <= r2;
    }

    // Bit u of the result: candidate q0 + u of the row (u < n <= 32) lies within the support. The
    // records of kQueryBatch candidates load together; those past the row's end are read (the record
    // arrays are padded by kRecordPad) and masked. `tiny` is set by hits with 0 < d2 < 2^-96.
    constexpr uint32_t kQueryBatch = 4;
    static_assert(kQueryBatch <= kRecordPad && 32u % kQueryBatch == 0u, "loads past the end of a row");

    __device__ __forceinline__ uint32_t hitMask(const float4* __restrict__ recs, const RowSpan& s, uint32_t q0, uint32_t n,
                                                float xi, float yi, float zi, float r2, bool& tiny)
    {
        uint32_t m = 0;
        for (uint32_t t = 0; t < n; t += kQueryBatch)
        {
            float4 p[kQueryBatch];
#pragma unroll
            for (uint32_t u = 0; u < kQueryBatch; u++) { p[u] = recs[s.at(q0 + t + u)]; }
#pragma unroll
            for (uint32_t u = 0; u < kQueryBatch; u++)
            {
                const float d2 = dist2(xi - p[u].x, yi - p[u].y, zi - p[u].z);
                const bool hit = d2 <= r2 && t + u < n;
                m |= (hit ? 1u : 0u) << (t + u);
                tiny = tiny || (hit && tinyDist2(d2));
            }
        }
        return m;
    }

    // The same for a whole row of at most 32 candidates, without the tiny test: the run's byte offset, the
    // distance in the reference's order, the compare and the mask are about eleven instructions per
    // candidate. Record offsets are 32-bit (kNearMax).
    constexpr uint32_t kNearBatch = 4;
    static_assert(kNearBatch <= kRecordPad && 32u % kNearBatch == 0u, "loads past the end of a row");
    constexpr uint32_t kNearMax = 1u << 27;      // most records for 32-bit byte offsets

    __device__ __forceinline__ uint32_t hitMaskNear(const float4* __restrict__ recs, const RowSpan& s, float xi, float yi,
                                                    float zi, float r2)
    {
        // (the second run's offset counts from the row's start and may lie up to 32 records below 0)
        const char* p = reinterpret_cast<const char*>(recs) - 32 * sizeof(float4);
        const uint32_t a = (s.oA + 32u) * static_cast<uint32_t>(sizeof(float4)), b = (s.oB + 32u) * static_cast<uint32_t>(sizeof(float4));
        uint32_t m = 0, t = 0;
        for (; t < s.n; t += kNearBatch, p += kNearBatch * sizeof(float4))
        {
            float v[kNearBatch][3];
#pragma unroll
            for (uint32_t u = 0; u < kNearBatch; u++)
            {
                const float* q = reinterpret_cast<const float*>(p + static_cast<size_t>(t + u < s.nA ? a : b) + u * sizeof(float4));
                v[u][0] = q[0]; v[u][1] = q[1]; v[u][2] = q[2];
            }
            __builtin_amdgcn_sched_barrier(0);   // (all loads of the batch before its first test)
            uint32_t four = 0;
#pragma unroll
            for (uint32_t u = 0; u < kNearBatch; u++)
            {
                const float d2 = dist2(xi - v[u][0], yi - v[u][1], zi - v[u][2]);
                four |= (d2 <= r2 ? 8u : 0u) >> u;
            }
            m = (m << 4) | four;
        }
        if (t == 0u) { return 0u; }
        m = __brev(m) >> (32u - t);   // candidate 0 came in first
        return s.n < 32u ? m & ((1u << s.n) - 1u) : m;
    }

    // A pair can only have 0 < d2 < 2^-96 if all its coordinate differences lie below 2^-48, one of
    // them nonzero; floats of magnitude 2^-23 and up differ by at least 2^-47. So only particles with a
    // coordinate nearer to zero than that are tested for such pairs.
    __device__ __forceinline__ bool mayBeTiny(const float4& p)
    {
        return fminf(fminf(__builtin_fabsf(p.x), __builtin_fabsf(p.y)), __builtin_fabsf(p.z)) < 0x1p-23f;
    }

    // reductions over the lanes of one SELL slice (a wave)
    __device__ __forceinline__ uint32_t sliceMax(uint32_t v)
    {
        for (int o = kSlice / 2; o > 0; o >>= 1) { v = max(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), o, kSlice))); }
        return v;
    }

    __device__ __forceinline__ uint32_t sliceMin(uint32_t v)
    {
        for (int o = kSlice / 2; o > 0; o >>= 1) { v = min(v, static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), o, kSlice))); }
        return v;
    }

    __device__ __forceinline__ uint32_t sliceSum(uint32_t v)
    {
        for (int o = kSlice / 2; o > 0; o >>= 1) { v += static_cast<uint32_t>(__shfl_xor(static_cast<int>(v), o, kSlice)); }
        return v;
    }

    // the rank of keys[t] (distinct values) among the 256 of the block, the largest first; all threads of
    // a block of 256 x kShare call it: each share counts a part of the keys. rank[] is zero before and
    // valid after the next barrier.
    template <uint32_t kShare>
    __device__ __forceinline__ void rankDown(const uint32_t* keys, uint32_t* rank)
    {
        const uint32_t t = threadIdx.x & (kBlock - 1u), part = threadIdx.x / kBlock;
        const uint32_t own = keys[t];
        const uint32_t lo = part * (kBlock / 4u) / kShare * 4u, hi = (part + 1u) * (kBlock / 4u) / kShare * 4u;
        uint32_t r = 0;
        for (uint32_t u = lo; u < hi; u += 4u)
        {
            const uint4 v = *reinterpret_cast<const uint4*>(&keys[u]);
            r += (v.x > own ? 1u : 0u) + (v.y > own ? 1u : 0u) + (v.z > own ? 1u : 0u) + (v.w > own ? 1u : 0u);
        }
        atomicAdd(&rank[t], r);
    }

    // The count pass (kShare: waves per 64 particles): hit masks, counts and index spans per particle; then the block's list positions,
    // slice headers and storage. Storage is taken from the pools with one atomic per block (the
    // blocks' order in the pools does not matter), so no scan over the slices follows.
    template <uint32_t kShare>
    __global__ void __launch_bounds__(kBlock * kShare) kQueryCount(Dev d)
    {
        __shared__ uint32_t cntS[3][kBlock], minS[3][kBlock], maxS[3][kBlock];
        __shared__ uint32_t openS[kBlock];       // kOpenF, kOpenB
        __shared__ __align__(16) uint32_t keyS[kBlock];
        __shared__ uint32_t rankS[kBlock];
        __shared__ uint32_t unitsS[3][kBlock / kSlice], entriesS[3][kBlock / kSlice];
        __shared__ uint32_t baseS[3];
        __shared__ uint8_t whoS[kBlock];
        const uint32_t blk = xcdBlock();
        const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
        const uint32_t local = (wave / kShare) * 64u + lane, share = wave % kShare;
        const uint32_t i = blk * kBlock + local;
        const uint32_t sc = uniformLoad(&d.blockScene[blk]);
        const Frame f = uniformLoad(&d.frames[sc]);
        const float r2 = uniformLoad(&d.consts[sc]).r2;
        if (threadIdx.x < kBlock)
        {
            for (int r = 0; r < 3; r++) { cntS[r][threadIdx.x] = 0u; minS[r][threadIdx.x] = kEmpty32; maxS[r][threadIdx.x] = 0u; }
            openS[threadIdx.x] = 0u;
            rankS[threadIdx.x] = 0u;
        }
        const bool active = keyAt(d, d.keyF, i) < f.emptyKey;
        const float4 pi = d.pos[i];
        __syncthreads();
        const bool masks = f.reach == 1;
        const Stencil s = stencilOf<kShare>(f, pi, active, share);
        const bool quick = !__any(active && mayBeTiny(pi)) && max(d.nF, d.nB) < kNearMax;
        uint32_t cnt[2] = { 0, 0 }, mn[2] = { kEmpty32, kEmpty32 }, mx[2] = { 0, 0 };
        uint32_t open = 0;
        bool tiny = false;
        // the wave's rows, fluid then boundary; the next row's cells load while the current one is tested
        RowCells next = s.cells(d.cellF, s.first, active);
#pragma unroll 1
        for (uint32_t row = s.first, rel = 0; row < s.last;)
        {
            const RowSpan w = next.span();
            const uint32_t nextRel = rel ^ 1u, nextRow = row + rel;
            if (nextRow < s.last) { next = s.cells(nextRel ? d.cellB : d.cellF, nextRow, active); }
            const float4* recs = rel ? d.bpos : d.pos;
            uint32_t m = 0, n = 0, lo = kEmpty32, hi = 0;
            for (uint32_t q0 = 0; q0 < w.n; q0 += 32u)
            {
                m = (quick && w.n <= 32u) ? hitMaskNear(recs, w, pi.x, pi.y, pi.z, r2)
                                          : hitMask(recs, w, q0, min(32u, w.n - q0), pi.x, pi.y, pi.z, r2, tiny);
                if (m)
                {
                    n += static_cast<uint32_t>(__popc(m));
                    lo = min(lo, w.at(q0 + static_cast<uint32_t>(__ffs(static_cast<int>(m))) - 1u));
                    hi = max(hi, w.at(q0 + 31u - static_cast<uint32_t>(__clz(static_cast<int>(m)))));
                }
            }
            if (masks)
            {
                if (w.n > 32u) { open |= 1u << (row + (rel ? kOpenB : kOpenF)); }
                if (rel == 0u) { d.ffMask[static_cast<size_t>(row) * d.nF + i] = m; }
                else if (w.n) { d.fbMask[static_cast<size_t>(row) * d.nF + i] = m; }
            }
            const uint32_t r = rel;
            cnt[0] += r ? 0u : n; cnt[1] += r ? n : 0u;
            mn[0] = r ? mn[0] : min(mn[0], lo); mn[1] = r ? min(mn[1], lo) : mn[1];
            mx[0] = r ? mx[0] : max(mx[0], hi); mx[1] = r ? max(mx[1], hi) : mx[1];
            rel = nextRel; row = nextRow;
        }
        if (d.nR)
        {
#pragma unroll 1
            for (uint32_t row = s.first; row < s.last; row++)
            {
                const RowSpan w = s.cells(d.cellR, row, active).span();
                for (uint32_t q = 0; q < w.n; q++)
                {
                    const uint32_t j = d.idxR[w.at(q)];
                    if (within(pi.x, pi.y, pi.z, d.rpos[j], r2))
                    {
                        atomicAdd(&cntS[2][local], 1u); atomicMin(&minS[2][local], j); atomicMax(&maxS[2][local], j);
                    }
                }
            }
        }
        if (tiny) { atomicOr(&d.status->pairTiny, 1u); }
        for (int r = 0; r < 2; r++)
        {
            if (cnt[r]) { atomicAdd(&cntS[r][local], cnt[r]); atomicMin(&minS[r][local], mn[r]); atomicMax(&maxS[r][local], mx[r]); }
        }
        if (open) { atomicOr(&openS[local], open); }
        __syncthreads();
        // thread t < 256: particle t of the block
        const uint32_t t = threadIdx.x, me = blk * kBlock + t;
        uint32_t c[3] = { 0, 0, 0 }, lo[3] = { kEmpty32, kEmpty32, kEmpty32 }, hi[3] = { 0, 0, 0 };
        if (t < kBlock)
        {
            for (int r = 0; r < 3; r++) { c[r] = cntS[r][t]; lo[r] = minS[r][t]; hi[r] = maxS[r][t]; }
            const bool wide = c[0] > 0 && hi[0] - lo[0] > 0xffffu;
            d.ffMask[static_cast<size_t>(kMaskRows) * d.nF + me] = masks ? openS[t] : 0xffffffffu;
            d.cnt[REL_FF][me] = static_cast<uint16_t>(c[0]);
            d.cnt[REL_FB][me] = static_cast<uint16_t>(c[1]);
            d.cnt[REL_FR][me] = static_cast<uint16_t>(c[2]);
            d.ffMin[me] = (c[0] > 0 ? lo[0] : 0u) | (wide ? kWideBit : 0u);
            // u16 counts, as the reference's (neighbor_lists.h:43)
            if (c[0] > 0xffffu || c[1] > 0xffffu || c[2] > 0xffffu) { atomicOr(&d.status->overflow, 2u); }
            // the block's list positions, longest lists first (ties in particle order): the keys are
            // made distinct by the thread index in their low byte
            keyS[t] = (min(c[0], 255u) << 8) | (kBlock - 1u - t);
        }
        __syncthreads();
        rankDown<kShare>(keyS, rankS);
        __syncthreads();
        if (t < kBlock)
        {
            const uint32_t rank = rankS[t];
            d.laneRank[me] = static_cast<uint8_t>(rank);
            whoS[rank] = static_cast<uint8_t>(t);
            for (int r = 0; r < 3; r++) { cntS[r][rank] = c[r]; minS[r][rank] = lo[r]; maxS[r][rank] = hi[r]; }
        }
        __syncthreads();
        SliceMeta m[3];
        if (t < kBlock)
        {
            for (int r = 0; r < 3; r++) { c[r] = cntS[r][t]; lo[r] = minS[r][t]; hi[r] = maxS[r][t]; }
            d.head[me] = make_uint2((c[0] & 0xffffu) | (c[1] << 16), (c[2] & 0xffffu) | (static_cast<uint32_t>(whoS[t]) << 16));
            // per slice (a wave's 64 list positions): pitch, base (min index), format, entries
            for (int r = 0; r < 3; r++)
            {
                const uint32_t pitch = sliceMax(c[r]);
                const uint32_t smin = sliceMin(lo[r]);
                const uint32_t smax = sliceMax(hi[r]);
                const uint32_t sum = sliceSum(c[r]);
                const bool delta = pitch == 0 || smax - smin <= 0xffffu;
                m[r].pitch = static_cast<uint16_t>(pitch);
                m[r].format = delta ? kFmtDelta16 : kFmtAbs32;
                m[r].base = (pitch == 0 || !delta) ? 0u : smin;
                m[r].offset = pitch * kSlice * (delta ? 1u : 2u);
                m[r].entries = sum;
                if (lane == 0u) { unitsS[r][wave] = m[r].offset; entriesS[r][wave] = sum; }
            }
        }
        __syncthreads();
        if (t < 6u)
        {
            // storage of the block's slices and their entries, counted in 64 bits (the host refuses a
            // pool beyond 2^32 units and regrows one that is too small, before any list is written)
            static_assert(offsetof(Status, entries) == offsetof(Status, poolUnits) + 3 * sizeof(uint64_t), "one row of counters");
            const uint32_t r = t % 3u;
            const uint32_t* v = t < 3u ? unitsS[r] : entriesS[r];
            unsigned long long sum = 0;
            for (uint32_t q = 0; q < kBlock / kSlice; q++) { sum += v[q]; }
            const unsigned long long at = atomicAdd(reinterpret_cast<unsigned long long*>(d.status->poolUnits) + t, sum);
            if (t < 3u) { baseS[r] = static_cast<uint32_t>(at); }
        }
        __syncthreads();
        if (t < kBlock && lane == 0u)
        {
            for (int r = 0; r < 3; r++)
            {
                uint32_t o = baseS[r];
                for (uint32_t q = 0; q < wave; q++) { o += unitsS[r][q]; }
                m[r].offset = o;
                d.meta[r][me / kSlice] = m[r];
            }
        }
    }

    // The fill pass: the lists of a block from the count pass's hit masks (rows they do not cover are
    // tested again), and the block's FF halo: the distinct FF neighbors of its particles, ascending.
    // With a halo (at most kHaloMax particles) the FF entries are slots of it, so the solver kernels
    // stage the neighbor records in LDS once per block; otherwise they are particle indices.
    //
    // The halo is a bitmap in LDS over pages of 256 particles, found through a small hash table: a
    // block's neighbors are runs of the sorted particles in at most about 40 pages. Each run's hit mask
    // goes into the bitmap whole (two words at most). Ranking the pages orders it, and the bitmap is
    // then spread into a table of halo slots, one per particle of the pages in page order, so that an
    // entry is one LDS read at its run's base plus its candidate number. The entries are staged in LDS
    // by list position and leave as whole slice rows.
    //
    // FF lists that span more than 0xffff indices keep the DictDelta16x2 order of the reference's
    // per-particle dict chunks (neighbor_lists.cpp:838-858): the neighbors within 0xffff of the
    // smallest form the low group, the rest the high group, which is stored from the back when it fits
    // 0xffff itself, else the candidate order stays; a list of more than kDictMax entries is no dict
    // (candidate order).
    // One kernel in place of the fill, the wide lists' fill and a halo kernel that read all entries back
    // twice (hash set and sort in LDS): 1M cube drop 352 to 205 us, 8M dam break 2,551 to 1,439 us, 64k
    // dam break 80 to 37 us, 4k 78 to 36 us. It is bound by its chain of phases (two blocks per CU for
    // the 66 KB of LDS) and the divergence of the loops over hits.
    constexpr uint32_t kStage = 40;          // FF entries per list staged in LDS; the rest are stored directly
    constexpr uint32_t kPages = 64;          // pages of a halo
    constexpr uint32_t kPageSlots = 128;     // slots of their hash table
    constexpr uint32_t kPageBits = 8;
    constexpr uint32_t kPageWords = (1u << kPageBits) / 32u;

    __device__ __forceinline__ uint32_t pageHash(uint32_t page) { return (page * 2654435761u) >> 25; }
    static_assert(kPageSlots == 1u << 7, "pageHash gives seven bits");

    __global__ void __launch_bounds__(kQueryThreads) __attribute__((amdgpu_waves_per_eu(6))) kQueryFill(Dev d)
    {
        if (stopped(d)) { return; }
        __shared__ uint16_t stage[kStage][kBlock];
        __shared__ __align__(16) uint16_t slotOf[kPages << kPageBits];   // halo entry of each particle of the pages
        __shared__ uint32_t bits[kPageSlots * kPageWords];
        __shared__ __align__(16) uint32_t pageKey[kPageSlots];     // page number + 1, 0: free
        __shared__ uint32_t pageRank[kPageSlots], pageBase[kPages];
        __shared__ uint32_t partF[kQueryShare][kBlock], partB[kQueryShare][kBlock];
        __shared__ uint32_t base2S[kBlock], maxRefS[kBlock];
        __shared__ uint32_t failS, pagesS, countS;
        const uint32_t blk = xcdBlock();
        const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
        const uint32_t local = (wave / kQueryShare) * 64u + lane, share = wave % kQueryShare;
        const uint32_t i = blk * kBlock + local;
        const uint32_t sc = uniformLoad(&d.blockScene[blk]);
        const Frame f = uniformLoad(&d.frames[sc]);
        const float r2 = uniformLoad(&d.consts[sc]).r2;
        for (uint32_t q = t; q < kPageSlots * kPageWords; q += kQueryThreads) { bits[q] = 0u; }
        if (t < kPageSlots) { pageKey[t] = 0u; pageRank[t] = 0u; }
        if (t < kPages) { pageBase[t] = 0u; }
        if (t < kBlock) { base2S[t] = kEmpty32; maxRefS[t] = 0u; }
        if (t == 0) { failS = 0u; pagesS = 0u; }
        const bool active = keyAt(d, d.keyF, i) < f.emptyKey;
        const float4 pi = d.pos[i];
        const uint32_t nF = active ? d.cnt[REL_FF][i] : 0u, nB = active ? d.cnt[REL_FB][i] : 0u, nR = active ? d.cnt[REL_FR][i] : 0u;
        const uint32_t fMin = d.ffMin[i];
        const uint32_t open = d.ffMask[static_cast<size_t>(kMaskRows) * d.nF + i];
        const uint32_t pos = blk * kBlock + d.laneRank[i];
        const uint32_t col = pos & (kBlock - 1u), lw = pos & (kSlice - 1u);
        const bool masks = f.reach == 1;
        const Stencil s = stencilOf<kQueryShare>(f, pi, active, share);
        bool ignored = false;
        // fn(row span, first candidate, hits) for up to 32 candidates at a time of the wave's rows, in list
        // order. Three rows inside the frame load their cells and masks at once.
        const auto each = [&](int rel, bool need, auto&& fn)
        {
            const uint2* table = rel == 0 ? d.cellF : d.cellB;
            const uint32_t* mask = rel == 0 ? d.ffMask : d.fbMask;
            const uint32_t opens = masks ? open >> (rel == 0 ? kOpenF : kOpenB) : 0xffffffffu;
            const auto take = [&](const RowSpan& w, uint32_t row, uint32_t m)
            {
                const bool covered = masks && ((opens >> row) & 1u) == 0u;
                for (uint32_t q0 = 0; q0 < w.n; q0 += 32u)
                {
                    if (!covered) { m = hitMask(rel == 0 ? d.pos : d.bpos, w, q0, min(32u, w.n - q0), pi.x, pi.y, pi.z, r2, ignored); }
                    if (m) { fn(w, q0, m); }
                }
            };
            if (s.near)
            {
                RowCells c[kMaskRows / kQueryShare];
                uint32_t m[kMaskRows / kQueryShare];
#pragma unroll
                for (uint32_t u = 0; u < kMaskRows / kQueryShare; u++)
                {
                    c[u] = s.cells(table, s.first + u, need);
                    m[u] = mask[static_cast<size_t>(s.first + u) * d.nF + i];
                }
#pragma unroll
                for (uint32_t u = 0; u < kMaskRows / kQueryShare; u++) { take(c[u].span(), s.first + u, m[u]); }
                return;
            }
#pragma unroll 1
            for (uint32_t row = s.first; row < s.last; row++)
            {
                take(s.cells(table, row, need).span(), row, masks ? mask[static_cast<size_t>(row) * d.nF + i] : 0u);
            }
        };
        // the hits of the two runs of a row: fn(first particle of the run's hits, hits from it, its candidate)
        const auto runs = [&](const RowSpan& w, uint32_t q0, uint32_t m, auto&& fn)
        {
            const uint32_t nA = w.nA > q0 ? min(w.nA - q0, 32u) : 0u;
            const uint32_t mA = nA < 32u ? m & ((1u << nA) - 1u) : m;
#pragma unroll
            for (uint32_t part = 0; part < 2u; part++)
            {
                const uint32_t h = part ? m ^ mA : mA;
                if (h) { const uint32_t q = static_cast<uint32_t>(__ffs(static_cast<int>(h))) - 1u; fn(q0 + q + (part ? w.oB : w.oA), h >> q, q); }
            }
        };
        const bool wide = (fMin & kWideBit) != 0u;
        const uint32_t minRef = fMin & ~kWideBit;
        const bool dict = wide && nF <= kDictMax;
        // the hash slot of a page; a table that is full gives up on the halo (failS)
        const auto pageSlot = [&](uint32_t page)
        {
            uint32_t h = pageHash(page);
            for (uint32_t probes = 0; probes < kPageSlots; probes++)
            {
                uint32_t v = __hip_atomic_load(&pageKey[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (v == 0u)
                {
                    v = atomicCAS(&pageKey[h], 0u, page + 1u);
                    if (v == 0u) { atomicAdd(&pagesS, 1u); return h; }
                }
                if (v == page + 1u) { return h; }
                h = (h + 1u) & (kPageSlots - 1u);
            }
            failS = 1u;
            return h;
        };
        __syncthreads();
        // the wave's neighbors: into the bitmap, and counted (a dict list's high group apart), so that
        // the next waves know where their part of each list starts
        {
            uint32_t n = 0, high = 0;
            each(0, nF != 0u, [&](const RowSpan& w, uint32_t q0, uint32_t m)
            {
                n += static_cast<uint32_t>(__popc(m));
                runs(w, q0, m, [&](uint32_t j, uint32_t h, uint32_t)
                {
                    if (dict)
                    {
                        const uint32_t jMax = j + 31u - static_cast<uint32_t>(__clz(static_cast<int>(h)));
                        atomicMax(&maxRefS[local], jMax);
                        if (jMax - minRef > 0xffffu)
                        {
                            // the first hit of the run beyond the low group
                            const uint32_t skip = j - minRef > 0xffffu ? 0u : minRef + 0x10000u - j;
                            const uint32_t hh = h >> skip;
                            high += static_cast<uint32_t>(__popc(hh));
                            atomicMin(&base2S[local], j + skip + static_cast<uint32_t>(__ffs(static_cast<int>(hh))) - 1u);
                        }
                    }
                    const uint32_t word = (j >> 5) & (kPageWords - 1u), sh = j & 31u;
                    const uint32_t slot = pageSlot(j >> kPageBits);
                    atomicOr(&bits[slot * kPageWords + word], h << sh);
                    const uint32_t rest = sh ? h >> (32u - sh) : 0u;
                    if (rest)
                    {
                        const uint32_t next = word + 1u < kPageWords ? slot * kPageWords + word + 1u : pageSlot((j >> kPageBits) + 1u) * kPageWords;
                        atomicOr(&bits[next], rest);
                    }
                });
            });
            partF[share][local] = (n - high) | (high << 16);
            uint32_t nb = 0;
            if (__any(nB != 0u)) { each(1, nB != 0u, [&](const RowSpan&, uint32_t, uint32_t m) { nb += static_cast<uint32_t>(__popc(m)); }); }
            partB[share][local] = nb;
        }
        __syncthreads();
        // pages in ascending order: their ranks, then the halo slots where they start
        const bool fits = !failS && pagesS <= kPages;
        if (fits && t < 4u * kPageSlots)
        {
            const uint32_t p = t & (kPageSlots - 1u), part = t / kPageSlots;
            const uint32_t own = pageKey[p];
            uint32_t r = 0;
            for (uint32_t u = part * (kPageSlots / 4u); u < (part + 1u) * (kPageSlots / 4u); u += 4u)
            {
                // (free slots hold 0 and sort last: 0 - 1 is the largest)
                const uint4 v = *reinterpret_cast<const uint4*>(&pageKey[u]);
                r += (v.x - 1u < own - 1u ? 1u : 0u) + (v.y - 1u < own - 1u ? 1u : 0u) + (v.z - 1u < own - 1u ? 1u : 0u)
                     + (v.w - 1u < own - 1u ? 1u : 0u);
            }
            if (own) { atomicAdd(&pageRank[p], r); }
        }
        __syncthreads();
        if (fits && t < kPageSlots && pageKey[t])
        {
            uint32_t n = 0;
            for (uint32_t w = 0; w < kPageWords; w++) { n += static_cast<uint32_t>(__popc(bits[t * kPageWords + w])); }
            pageBase[pageRank[t]] = n;
        }
        __syncthreads();
        if (t < kPages)
        {
            const uint32_t own = pageBase[t];
            uint32_t incl = own;
            for (int o = 1; o < 64; o <<= 1)
            {
                const uint32_t v = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), o, 64));
                if (lane >= static_cast<uint32_t>(o)) { incl += v; }
            }
            pageBase[t] = incl - own;
            if (t == kPages - 1u)
            {
                countS = (!fits || incl > kHaloMax) ? kNoHalo : incl;
                d.haloInfo[blk] = HaloInfo{ countS, 1u };
            }
        }
        static_assert(kPages == 64, "the page counts are scanned by one wave");
        __syncthreads();
        const bool halo = countS != kNoHalo;
        if (halo)
        {
            // one word of the bitmap per thread: its particles into the halo, its slots into the table
            uint32_t* out = d.haloIdx + static_cast<size_t>(blk) * kHaloMax;
            for (uint32_t q = t; q < kPageSlots * kPageWords; q += kQueryThreads)
            {
                uint32_t b = bits[q];
                if (b == 0u) { continue; }
                const uint32_t p = q / kPageWords, w = q & (kPageWords - 1u);
                const uint32_t rank = pageRank[p];
                uint32_t r = pageBase[rank];
                for (uint32_t v = 0; v < w; v++) { r += static_cast<uint32_t>(__popc(bits[p * kPageWords + v])); }
                const uint32_t j0 = ((pageKey[p] - 1u) << kPageBits) + 32u * w;
                uint16_t* table = slotOf + (rank << kPageBits) + 32u * w;
                while (b)
                {
                    const uint32_t u = static_cast<uint32_t>(__ffs(static_cast<int>(b))) - 1u;
                    out[r] = j0 + u;
                    table[u] = static_cast<uint16_t>(r << kSlotShift);
                    r++;
                    b &= b - 1u;
                }
            }
            __syncthreads();
        }
        // the entries: FF by slot or index, FB and FR by index
        uint32_t low = 0, high = 0, kB = 0;
        for (uint32_t q = 0; q < share; q++) { const uint32_t v = partF[q][local]; low += v & 0xffffu; high += v >> 16; kB += partB[q][local]; }
        const bool split = dict && maxRefS[local] - base2S[local] <= 0xffffu;
        if (!split) { low += high; }
        {
            const SliceMeta mF = d.meta[REL_FF][pos / kSlice];
            uint16_t* rows = d.pool[REL_FF] + mF.offset + lw;
            each(0, nF != 0u, [&](const RowSpan& w, uint32_t q0, uint32_t m)
            {
                // table positions of the runs' candidates: the run's first hit is in the table, and the
                // page after its own, when the run has hits there, is the next in the table
                uint32_t tA = 0, tB = 0;
                if (halo)
                {
                    runs(w, q0, m, [&](uint32_t j, uint32_t, uint32_t q)
                    {
                        uint32_t h = pageHash(j >> kPageBits);
                        for (uint32_t probes = 0; probes < kPageSlots && pageKey[h] != (j >> kPageBits) + 1u; probes++) { h = (h + 1u) & (kPageSlots - 1u); }
                        const uint32_t at = (pageRank[h] << kPageBits) + (j & ((1u << kPageBits) - 1u)) - q;
                        if (q0 + q < w.nA) { tA = at; } else { tB = at; }
                    });
                }
                while (m)
                {
                    const uint32_t q = static_cast<uint32_t>(__ffs(static_cast<int>(m))) - 1u;
                    m &= m - 1u;
                    const uint32_t j = w.at(q0 + q);
                    const uint32_t k = (split && j - minRef > 0xffffu) ? nF - ++high : low++;
                    if (halo)
                    {
                        const uint16_t e = slotOf[q + (q0 + q < w.nA ? tA : tB)];
                        if (k < kStage) { stage[k][col] = e; } else { rows[k * kSlice] = e; }
                    }
                    else { sellWrite(d.pool[REL_FF], mF, lw, k, j); }
                }
            });
        }
        if (__any(nB != 0u))
        {
            const SliceMeta mB = d.meta[REL_FB][pos / kSlice];
            each(1, nB != 0u, [&](const RowSpan& w, uint32_t q0, uint32_t m)
            {
                while (m)
                {
                    const uint32_t q = static_cast<uint32_t>(__ffs(static_cast<int>(m))) - 1u;
                    m &= m - 1u;
                    sellWrite(d.pool[REL_FB], mB, lw, kB++, w.at(q0 + q));
                }
            });
        }
        if (nR && share == 0u)
        {
            // few particles have rigid neighbors: one wave walks their rows
            const SliceMeta mR = d.meta[REL_FR][pos / kSlice];
            uint32_t kR = 0;
#pragma unroll 1
            for (uint32_t r = 0; r < s.side * s.side * s.chunks; r++)
            {
                const RowSpan w = s.cells(d.cellR, r, true).span();
                for (uint32_t q = 0; q < w.n; q++)
                {
                    const uint32_t j = d.idxR[w.at(q)];
                    if (within(pi.x, pi.y, pi.z, d.rpos[j], r2)) { sellWrite(d.pool[REL_FR], mR, lw, kR++, j); }
                }
            }
        }
        if (!halo) { return; }
        __syncthreads();
        // the staged entries leave as whole slice rows; the slices of a block with a halo are u16 slices
        const uint32_t p = t & (kBlock - 1u);
        SliceMeta& m = d.meta[REL_FF][(blk * kBlock + p) / kSlice];
        const uint32_t n = min(static_cast<uint32_t>(d.head[blk * kBlock + p].x & 0xffffu), kStage);
        uint16_t* row = d.pool[REL_FF] + m.offset + (p & (kSlice - 1u));
        for (uint32_t k = t / kBlock; k < n; k += kQueryShare) { row[k * kSlice] = stage[k][p]; }
        if (t < kBlock && (t & (kSlice - 1u)) == 0u) { m.format = kFmtDelta16; }
    }

    // ----------------------------------------------------------------------------------------
    // rigid-source lists, one wave per rigid particle: mode 0 counts RF, RB and RR; mode 1 fills
    // the RF CSR; mode 2 fills RF and the RB and RR lists of the contact solver. The candidates of
    // a relation -- cell by cell in z-y-x order, by index inside a cell -- are tested 64 at a
    // time, and ballots keep that order in the lists.

    __global__ void __launch_bounds__(kBlock) kQueryRigid(Dev d, int mode)
    {
        if (stopped(d)) { return; }
        const uint32_t i = (blockIdx.x * kBlock + threadIdx.x) >> 6;
        const uint32_t lane = threadIdx.x & 63u;
        if (i >= d.nR) { return; }
        const bool fill = mode != 0;
        const bool contact = mode == 2;
        const uint32_t sc = d.bodyScene[d.rbody[i]];
        const Frame& f = d.frames[sc];
        const float r2 = d.consts[sc].r2;
        const int reach = f.reach;
        const float4 pi = d.rpos[i];
        const int cx = floorToInt(pi.x * f.cellSizeInv) - f.orig[0];
        const int cy = floorToInt(pi.y * f.cellSizeInv) - f.orig[1];
        const int cz = floorToInt(pi.z * f.cellSizeInv) - f.orig[2];
        uint32_t cnt[3] = { 0, 0, 0 };
        uint32_t w[3] = { fill ? d.rfOff[i] : 0u, contact ? d.rbOff[i] : 0u, contact ? d.rrOff[i] : 0u };
        const bool inside = cx >= 0 && cx < static_cast<int>(f.dim[0]) && cy >= 0 && cy < static_cast<int>(f.dim[1])
                         && cz >= 0 && cz < static_cast<int>(f.dim[2]);
        if (inside)
        {
            const int lo[3] = { max(cx - reach, 0), max(cy - reach, 0), max(cz - reach, 0) };
            const int hi[3] = { min(cx + reach, static_cast<int>(f.dim[0]) - 1), min(cy + reach, static_cast<int>(f.dim[1]) - 1),
                                min(cz + reach, static_cast<int>(f.dim[2]) - 1) };
            const uint32_t nx = static_cast<uint32_t>(hi[0] - lo[0] + 1), ny = static_cast<uint32_t>(hi[1] - lo[1] + 1);
            const uint32_t nCells = nx * ny * static_cast<uint32_t>(hi[2] - lo[2] + 1);
            const uint32_t body = d.rbody[i];
            const uint64_t below = (1ull << lane) - 1ull;
            const int nRel = (fill && !contact) ? 1 : 3;
            for (uint32_t c0 = 0; c0 < nCells; c0 += 64)
            {
                // this lane's cell of the batch and its three ranges
                const uint32_t c = c0 + lane;
                uint2 rng[3] = { make_uint2(0u, 0u), make_uint2(0u, 0u), make_uint2(0u, 0u) };
                if (c < nCells)
                {
                    const uint32_t lin = linearCell(f, lo[0] + static_cast<int>(c % nx), lo[1] + static_cast<int>((c / nx) % ny),
                                                    lo[2] + static_cast<int>(c / (nx * ny)));
                    rng[0] = d.cellF[lin];
                    rng[1] = d.cellB[lin];
                    if (d.nR) { rng[2] = d.cellR[lin]; }
                }
                for (int rel = 0; rel < nRel; rel++)
                {
                    // inclusive prefix of the cells' candidate counts over the lanes
                    const uint32_t size = rng[rel].y - rng[rel].x;
                    uint32_t incl = size;
                    for (int o = 1; o < 64; o <<= 1)
                    {
                        const uint32_t v = static_cast<uint32_t>(__shfl_up(static_cast<int>(incl), o, 64));
                        if (lane >= static_cast<uint32_t>(o)) { incl += v; }
                    }
                    const uint32_t total = static_cast<uint32_t>(__shfl(static_cast<int>(incl), 63, 64));
                    for (uint32_t f0 = 0; f0 < total; f0 += 64)
                    {
                        const uint32_t fi = f0 + lane;
                        bool hit = false;
                        uint32_t j = 0;
                        // the lane (cell) whose prefix range holds fi: the first with incl > fi
                        // (six halvings of [0, 63], taken by every lane together)
                        uint32_t a = 0, b = 63;
                        for (int step = 0; step < 6; step++)
                        {
                            const uint32_t m = (a + b) >> 1;
                            const uint32_t im = static_cast<uint32_t>(__shfl(static_cast<int>(incl), static_cast<int>(m), 64));
                            if (im > fi) { b = m; } else { a = m + 1; }
                        }
                        const uint32_t inclA = static_cast<uint32_t>(__shfl(static_cast<int>(incl), static_cast<int>(a), 64));
                        const uint32_t sizeA = static_cast<uint32_t>(__shfl(static_cast<int>(size), static_cast<int>(a), 64));
                        const uint32_t startA = static_cast<uint32_t>(__shfl(static_cast<int>(rng[rel].x), static_cast<int>(a), 64));
                        if (fi < total)
                        {
                            const uint32_t t = startA + (fi - (inclA - sizeA));
                            if (rel == 0) { j = t; hit = within(pi.x, pi.y, pi.z, d.pos[j], r2); }
                            else if (rel == 1) { j = t; hit = within(pi.x, pi.y, pi.z, d.bpos[j], r2); }
                            else
                            {
                                j = d.idxR[t];
                                hit = j != i && d.rbody[j] != body && within(pi.x, pi.y, pi.z, d.rpos[j], r2);
                            }
                        }
                        const uint64_t bal = __ballot(hit);
                        const bool store = rel == 0 ? fill : contact;
                        if (store && hit)
                        {
                            uint32_t* dst = rel == 0 ? d.rfIdx : (rel == 1 ? d.rbIdx : d.rrIdx);
                            dst[w[rel] + static_cast<uint32_t>(__popcll(bal & below))] = j;
                        }
                        const uint32_t n = static_cast<uint32_t>(__popcll(bal));
                        w[rel] += n;
                        cnt[rel] += n;
                    }
                }
            }
        }
        if (!fill && lane == 0)
        {
            if (i == 0) { d.rfOff[d.nR] = 0u; }
            d.rfCnt[i] = cnt[0];
            d.rfOff[i] = cnt[0];
            d.rbCnt[i] = cnt[1];
            d.rrCnt[i] = cnt[2];
        }
    }

    // totals of the rigid-source relations and the RF capacity check (after the RF offset scan);
    // a scene whose rigid particles have RB or RR entries runs the contact solve
    // (BuildRigidBoundaryNeighbors, rigid_solver.cpp:90-149)
    __global__ void __launch_bounds__(kBlock) kRigidTotals(Dev d)
    {
        __shared__ uint32_t red[2][kBlock];
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i < d.nR && (d.rbCnt[i] | d.rrCnt[i]) != 0u)
        {
            d.solve[d.bodyScene[d.rbody[i]]].contactActive = 1u;
        }
        red[0][threadIdx.x] = i < d.nR ? d.rbCnt[i] : 0u;
        red[1][threadIdx.x] = i < d.nR ? d.rrCnt[i] : 0u;
        __syncthreads();
        for (uint32_t o = kBlock / 2; o > 0; o >>= 1)
        {
            if (threadIdx.x < o) { red[0][threadIdx.x] += red[0][threadIdx.x + o]; red[1][threadIdx.x] += red[1][threadIdx.x + o]; }
            __syncthreads();
        }
        if (threadIdx.x == 0)
        {
            atomicAdd(reinterpret_cast<unsigned long long*>(&d.status->rbTotal), static_cast<unsigned long long>(red[0][0]));
            atomicAdd(reinterpret_cast<unsigned long long*>(&d.status->rrTotal), static_cast<unsigned long long>(red[1][0]));
        }
        if (i == 0)
        {
            d.status->rfTotal = d.rfOff[d.nR];
            if (d.rfOff[d.nR] > d.rfCap) { atomicOr(&d.status->overflow, 4u); }
        }
    }

    // the decision point of a captured step, after the search's counts and scans: what the host
    // would otherwise read to grow storage, rebuild a frame or take the contact solve calls off
    // the rest of the captured step (status->stop bit 1); the host then runs the step anew
    __global__ void kStepGate(Dev d)
    {
        if (threadIdx.x != 0) { return; }
        const Status& st = *d.status;
        bool grow = false;
        for (int r = 0; r < 3; r++) { grow = grow || st.poolUnits[r] > d.poolCap[r]; }
        const bool refuse = st.abort != 0u || st.overflow != 0u || grow || st.rbTotal != 0ull || st.rrTotal != 0ull
                            || (st.pairTiny != 0u && d.fastPairs != 0u);
        if (refuse) { d.status->stop |= 1u; }
    }

    // after the captured sweeps: a scene with fluid that has not converged calls off the captured
    // tail (bit 2); the host adds sweeps and runs the tail itself
    __global__ void __launch_bounds__(kBlock) kSolveGate(Dev d)
    {
        if (stopped(d)) { return; }
        bool open = false;
        for (uint32_t sc = threadIdx.x; sc < d.nScenes; sc += kBlock)
        {
            open = open || (d.scenes[sc].nF != 0u && d.solve[sc].converged == 0u);
        }
        if (open) { atomicOr(&d.status->stop, 2u); }
    }

    __global__ void kClearStop(Dev d)
    {
        if (threadIdx.x == 0) { d.status->stop = 0u; }
    }

    // scene AABB of the positions of one particle class (ComputeSceneAABB_ParticleClass,
    // neighbor_search.cpp:227-258); min/max are exact in any order
    __device__ __forceinline__ uint32_t orderedBits(float v)
    {
        const uint32_t u = __float_as_uint(v);
        return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    }

    // per-scene bounds of one population: out[6 s + a] holds the ordered bits of the min x, y, z
    // and then the max. Each wave walks a contiguous range of 64-particle chunks, keeps per-lane
    // running bounds while the chunks belong to one scene, and reduces them into that scene's
    // bounds with one set of atomics when the scene changes or the range ends (chunks that mix
    // scenes update lane by lane)
    __global__ void __launch_bounds__(kBlock) kAabb(Dev d, int pop, const float4* __restrict__ p, uint32_t n,
        uint32_t* __restrict__ out)
    {
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t nWaves = gridDim.x * (kBlock / 64);
        const uint32_t gw = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
        const uint32_t nChunks = (n + 63u) / 64u;
        const uint32_t c0 = static_cast<uint32_t>(static_cast<uint64_t>(nChunks) * gw / nWaves);
        const uint32_t c1 = static_cast<uint32_t>(static_cast<uint64_t>(nChunks) * (gw + 1) / nWaves);
        uint32_t rs = 0xffffffffu;
        uint32_t v[6] = { 0xffffffffu, 0xffffffffu, 0xffffffffu, 0u, 0u, 0u };
        const auto flush = [&]()
        {
            for (int o = 32; o > 0; o >>= 1)
            {
                for (int a = 0; a < 3; a++)
                {
                    v[a] = min(v[a], static_cast<uint32_t>(__shfl_xor(static_cast<int>(v[a]), o, 64)));
                    v[3 + a] = max(v[3 + a], static_cast<uint32_t>(__shfl_xor(static_cast<int>(v[3 + a]), o, 64)));
                }
            }
            if (lane == 0 && rs != 0xffffffffu)
            {
                for (int a = 0; a < 3; a++) { atomicMin(&out[6 * rs + a], v[a]); atomicMax(&out[6 * rs + 3 + a], v[3 + a]); }
            }
            for (int a = 0; a < 3; a++) { v[a] = 0xffffffffu; v[3 + a] = 0u; }
        };
        for (uint32_t c = c0; c < c1; c++)
        {
            const uint32_t i = c * 64u + lane;
            bool valid = i < n;
            uint32_t sc = 0;
            if (valid)
            {
                sc = sceneOfParticle(d, pop, i);
                if (pop == POP_F && i - d.scenes[sc].offF >= d.scenes[sc].nF) { valid = false; }
            }
            uint32_t b[3] = { 0, 0, 0 };
            if (valid)
            {
                const float4 q = p[i];
                b[0] = orderedBits(q.x); b[1] = orderedBits(q.y); b[2] = orderedBits(q.z);
            }
            const uint64_t vm = __ballot(valid);
            if (vm == 0) { continue; }
            const int first = __ffsll(static_cast<unsigned long long>(vm)) - 1;
            const uint32_t s0 = static_cast<uint32_t>(__shfl(static_cast<int>(sc), first, 64));
            if (__ballot(valid && sc != s0) == 0)
            {
                if (s0 != rs) { flush(); rs = s0; }
                if (valid)
                {
                    for (int a = 0; a < 3; a++) { v[a] = min(v[a], b[a]); v[3 + a] = max(v[3 + a], b[a]); }
                }
            }
            else if (valid)
            {
                for (int a = 0; a < 3; a++) { atomicMin(&out[6 * sc + a], b[a]); atomicMax(&out[6 * sc + 3 + a], b[a]); }
            }
        }
        flush();
    }

    // ----------------------------------------------------------------------------------------
    // host launchers

    static inline uint32_t blocksFor(uint64_t n) { return static_cast<uint32_t>((n + kBlock - 1) / kBlock); }

    // a sort of n keys runs as one block and uses no sort state
    bool radixSortSingleBlock(uint32_t n) { return n <= kSmallSort; }

    static uint32_t radixPasses(uint32_t bits) { return (bits + kRadixBits - 1u) / kRadixBits; }

    // cells: the cell tables hold the runs of the sorted keys, which are cleared
    void launchResetSearch(hipStream_t s, const Dev& d, bool cells)
    {
        const uint32_t nF = cells ? blocksFor(d.nF) : 0u, nR = cells ? blocksFor(d.nR) : 0u;
        kResetSearch<<<1u + nF + nR, kBlock, 0, s>>>(d, nF);
    }

    // key arrays hold u32 keys, or u64 keys (two words each) when d.key64
    // state: the sort state that takes the digit counts when kRadixPass sorts the keys by `bits` bits
    // (null: the keys are not sorted)
    void launchKeys(hipStream_t s, const Dev& d, int pop, const float4* p, uint32_t n, bool check, uint32_t* key,
                    uint32_t* idx, uint32_t bits, uint32_t* state)
    {
        if (!n) { return; }
        const uint32_t passes = state && !radixSortSingleBlock(n) && n <= kRadixSmallTiles ? radixPasses(bits) : 0u;
        const uint32_t nb = blocksFor(n);
        if (d.key64)
        {
            kKeys<<<nb, kBlock, 0, s>>>(d, pop, p, n, check, reinterpret_cast<uint64_t*>(key), idx, state, passes);
        }
        else { kKeys<<<nb, kBlock, 0, s>>>(d, pop, p, n, check, key, idx, state, passes); }
    }

    void launchKeysSorted(hipStream_t s, const Dev& d, const float4* p, uint32_t n, uint32_t* key, uint32_t* idx)
    {
        if (!n) { return; }
        if (d.key64) { kKeysSorted<<<blocksFor(n), kBlock, 0, s>>>(d, p, n, reinterpret_cast<uint64_t*>(key), idx); }
        else { kKeysSorted<<<blocksFor(n), kBlock, 0, s>>>(d, p, n, key, idx); }
    }

    template <typename K>
    static bool radixSort(hipStream_t s, K* key, uint32_t* idx, K* key2, uint32_t* idx2, uint32_t n, uint32_t bits,
                          uint32_t* state, uint32_t* fail, bool counted, bool copyBack)
    {
        if (n <= kSmallSort)
        {
            // fewer keys per lane leave fewer waves idle: 4,096 keys fill 16 waves with four each
            if (n <= kSmallThreads * 4u) { kSortSmall<K, 4><<<1, kSmallThreads, 0, s>>>(key, idx, n, bits); }
            else if (n <= kSmallThreads * 8u) { kSortSmall<K, 8><<<1, kSmallThreads, 0, s>>>(key, idx, n, bits); }
            else { kSortSmall<K, 16><<<1, kSmallThreads, 0, s>>>(key, idx, n, bits); }
            return false;
        }
        const uint32_t passes = radixPasses(bits);
        const bool few = n <= kRadixSmallTiles;
        const uint32_t nTiles = few ? (n + kRadixTileMin - 1) / kRadixTileMin : (n + kRadixManyTile - 1) / kRadixManyTile;
        if (few && !counted) { kRadixCount<K><<<blocksFor(n), kBlock, 0, s>>>(key, n, state, passes); }
        K* kIn = key; uint32_t* iIn = idx; K* kOut = key2; uint32_t* iOut = idx2;
        for (uint32_t q = 0; q < passes; q++)
        {
            if (few) { kRadixPass<K, kRadixPerMin><<<nTiles, kBlock, 0, s>>>(kIn, iIn, kOut, iOut, n, q, bits, state, fail); }
            else
            {
                uint32_t* totals = state + kRadixManyAt;
                uint32_t* hist = totals + kRadixBins;
                kRadixHist<K><<<nTiles, kBlock, 0, s>>>(kIn, n, q * kRadixBits, nTiles, hist);
                kRadixDigitScan<<<kRadixBins, kBlock, 0, s>>>(hist, nTiles, totals);
                kRadixScatter<K><<<nTiles, kBlock, 0, s>>>(kIn, iIn, kOut, iOut, n, q * kRadixBits, bits, nTiles, hist, totals);
            }
            K* t = kIn; kIn = kOut; kOut = t;
            uint32_t* ti = iIn; iIn = iOut; iOut = ti;
        }
        if (kIn == key) { return false; }
        if (!copyBack) { return true; }
        (void)hipMemcpyAsync(key, kIn, sizeof(K) * n, hipMemcpyDeviceToDevice, s);
        (void)hipMemcpyAsync(idx, iIn, sizeof(uint32_t) * n, hipMemcpyDeviceToDevice, s);
        return false;
    }

    // sorts (key, idx) stably by the low `bits` bits; state is a sort state of radixStateWords(n) words,
    // zeroed when allocated, fail its give-up word; counted: the keys come from launchKeys, which has added the digit
    // counts where they are needed. The
    // result ends in (key, idx), or, without copyBack, in (key2, idx2) after an odd number of passes:
    // the return value says which.
    bool launchRadixSort(hipStream_t s, bool key64, uint32_t* key, uint32_t* idx, uint32_t* key2, uint32_t* idx2,
                         uint32_t n, uint32_t bits, uint32_t* state, uint32_t* fail, bool counted, bool copyBack)
    {
        if (n < 2) { return false; }
        if (key64)
        {
            return radixSort(s, reinterpret_cast<uint64_t*>(key), idx, reinterpret_cast<uint64_t*>(key2), idx2, n, bits, state,
                             fail, counted, copyBack);
        }
        return radixSort(s, key, idx, key2, idx2, n, bits, state, fail, counted, copyBack);
    }

    void launchPermute(hipStream_t s, const Gather& g, const uint32_t* idx)
    {
        if (g.n) { kPermute<<<blocksFor(g.n), kBlock, 0, s>>>(g, idx); }
    }

    void launchPermuteCells(hipStream_t s, const Dev& d, const Gather& g)
    {
        if (g.n) { kPermuteCells<<<blocksFor(g.n), kBlock, 0, s>>>(d, g); }
    }

    void launchClearAll(hipStream_t s, uint2* cell, uint64_t n)
    {
        if (n) { kClearAll<<<blocksFor(n), kBlock, 0, s>>>(cell, n); }
    }

    void launchBuildCells(hipStream_t s, const Dev& d, const uint32_t* key, uint32_t n, uint2* cell)
    {
        if (n) { kBuildCells<<<blocksFor(n), kBlock, 0, s>>>(d, key, n, cell); }
    }

    void launchQueryCount(hipStream_t s, const Dev& d)
    {
        const uint32_t n = blocksFor(d.nF);
        if (n == 0u) { return; }
        if (n <= kShareBlocks) { kQueryCount<kQueryShare><<<n, kQueryThreads, 0, s>>>(d); }
        else { kQueryCount<1u><<<n, kBlock, 0, s>>>(d); }
    }

    void launchQueryFill(hipStream_t s, const Dev& d)
    {
        if (d.nF) { kQueryFill<<<blocksFor(d.nF), kQueryThreads, 0, s>>>(d); }
    }

    void launchQueryRigid(hipStream_t s, const Dev& d, int mode, uint32_t* tmp)
    {
        if (!d.nR) { return; }
        kQueryRigid<<<blocksFor(64ull * d.nR), kBlock, 0, s>>>(d, mode);
        if (mode == 0)
        {
            launchScan(s, d.rfOff, d.nR + 1, tmp, &d.status->scanFail);
            kRigidTotals<<<blocksFor(d.nR), kBlock, 0, s>>>(d);
        }
    }

    void launchStepGate(hipStream_t s, const Dev& d) { kStepGate<<<1, 64, 0, s>>>(d); }
    void launchSolveGate(hipStream_t s, const Dev& d) { kSolveGate<<<1, kBlock, 0, s>>>(d); }
    void launchClearStop(hipStream_t s, const Dev& d) { kClearStop<<<1, 64, 0, s>>>(d); }

    void launchAabb(hipStream_t s, const Dev& d, int pop, const float4* p, uint32_t n, uint32_t* out)
    {
        // about 8 chunks of 64 particles per wave, at most 256 blocks
        const uint32_t chunks = (n + 63u) / 64u;
        const uint32_t blocks = std::max(1u, std::min(256u, (chunks + 31u) / 32u));
        if (n) { kAabb<<<blocks, kBlock, 0, s>>>(d, pop, p, n, out); }
    }
}
