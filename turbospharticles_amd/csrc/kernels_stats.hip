// kernels_stats.hip -- per-scene statistics on the device (SimBackend_GPU::FillStatisticsRecord,
// GPU/backend/gpu_backend.cpp:1067-1208, statistics_kernels.cu): neighbor-count minimum, maximum
// and 99th percentile from an exact histogram of the counts, the averages of the relative density
// error rho/rho0 - 1 (raw, positive part, absolute), and the velocity magnitude's sum, minimum and
// maximum. A served scene is monitored without copying its particles to the host.
#include <mutex>

#include "tsp_device.h"

namespace tsp
{
    constexpr uint32_t kHistBins = 65536;   // neighbor counts are stored in 16 bits
    constexpr uint32_t kRelations = 6;      // FF, FB, FR (u16 counts), RF, RB, RR (u32)

    // the counts of one scene
    struct StatsCounts
    {
        const uint16_t* c16[3];
        const uint32_t* c32[3];
        uint32_t nF, nR;
    };

    // Histograms of all six relations' counts. Nearly all counts fall into a few dozen bins, so a global
    // atomic per particle runs at the rate of one address (4.7 ms per relation at 1M particles); each
    // block counts the low bins in LDS first and adds its nonzero ones (1M: all six in 20 us).
    constexpr uint32_t kLowBins = 512;

    __global__ void __launch_bounds__(kBlock) kStatsHist(StatsCounts c, uint32_t* __restrict__ hist)
    {
        __shared__ uint32_t low[kRelations][kLowBins];
        for (uint32_t q = threadIdx.x; q < kRelations * kLowBins; q += kBlock) { low[q / kLowBins][q % kLowBins] = 0u; }
        __syncthreads();
        const uint32_t stride = gridDim.x * kBlock;
        const auto count = [&](uint32_t r, uint32_t v)
        {
            if (v < kLowBins) { atomicAdd(&low[r][v], 1u); }
            else { atomicAdd(&hist[r * kHistBins + min(v, kHistBins - 1u)], 1u); }
        };
        for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < c.nF; i += stride)
        {
            for (uint32_t r = 0; r < 3u; r++) { count(r, c.c16[r][i]); }
        }
        for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < c.nR; i += stride)
        {
            for (uint32_t r = 0; r < 3u; r++) { count(3u + r, c.c32[r][i]); }
        }
        __syncthreads();
        for (uint32_t q = threadIdx.x; q < kRelations * kLowBins; q += kBlock)
        {
            const uint32_t v = low[q / kLowBins][q % kLowBins];
            if (v) { atomicAdd(&hist[(q / kLowBins) * kHistBins + q % kLowBins], v); }
        }
    }

    // Block r < 6: minimum, maximum and the value at sorted position (99 (n - 1)) / 100 of relation r's
    // histogram (ComputeStatsFromHistogram, statistics_kernels.cu:82-127), and the sum of its values.
    // Block 6: the fluid sums of kStatsFluid's partials. Chunks of 1024 bins: a wave sums four of them,
    // one wave scans the 64 chunk counts, then the chunk that holds the percentile (all in 13 us at 1M
    // particles; one thread scanning bins and partials took 6 x 46 + 843 us).
    constexpr uint32_t kScanThreads = 1024;
    constexpr uint32_t kChunk = 1024;
    constexpr uint32_t kChunks = kHistBins / kChunk;
    static_assert(kChunks == 64, "one wave scans the chunks");

    __device__ __forceinline__ uint32_t waveScan(uint32_t v)
    {
        for (int o = 1; o < 64; o <<= 1)
        {
            const uint32_t u = static_cast<uint32_t>(__shfl_up(static_cast<int>(v), o, 64));
            if ((threadIdx.x & 63u) >= static_cast<uint32_t>(o)) { v += u; }
        }
        return v;
    }

    __device__ void histogramStats(const uint32_t* __restrict__ hist, uint32_t n, uint64_t* __restrict__ out)
    {
        __shared__ uint32_t chunk[kChunks];
        __shared__ unsigned long long total;
        __shared__ uint32_t mn, mx;
        const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
        if (threadIdx.x == 0) { total = 0ull; mn = kHistBins; mx = 0u; }
        __syncthreads();
        unsigned long long sum = 0;
        uint32_t lo = kHistBins, hi = 0;
        for (uint32_t c = wave; c < kChunks; c += kScanThreads / 64u)
        {
            uint32_t s = 0;
            for (uint32_t q = 0; q < kChunk / 64u; q++)
            {
                const uint32_t v = c * kChunk + q * 64u + lane, h = hist[v];
                s += h;
                sum += static_cast<unsigned long long>(h) * v;
                if (h) { lo = min(lo, v); hi = max(hi, v); }
            }
            for (int o = 32; o > 0; o >>= 1) { s += static_cast<uint32_t>(__shfl_xor(static_cast<int>(s), o, 64)); }
            if (lane == 0u) { chunk[c] = s; }
        }
        if (hi || lo < kHistBins) { atomicAdd(&total, sum); atomicMin(&mn, lo); atomicMax(&mx, hi); }
        __syncthreads();
        if (wave != 0u) { return; }
        uint32_t p99 = 0;
        if (n > 0)
        {
            const uint32_t i99 = static_cast<uint32_t>((99ull * static_cast<uint64_t>(n - 1u)) / 100ull);
            const uint32_t incl = waveScan(chunk[lane]);
            const uint32_t c = static_cast<uint32_t>(__ffsll(static_cast<unsigned long long>(__ballot(incl > i99)))) - 1u;
            uint32_t before = c ? static_cast<uint32_t>(__shfl(static_cast<int>(incl), static_cast<int>(c) - 1, 64)) : 0u;
            for (uint32_t q = 0; q < kChunk / 64u; q++)
            {
                const uint32_t v = c * kChunk + q * 64u;
                const uint32_t in = before + waveScan(hist[v + lane]);
                const unsigned long long past = __ballot(in > i99);
                if (past) { p99 = v + static_cast<uint32_t>(__ffsll(past)) - 1u; break; }
                before = static_cast<uint32_t>(__shfl(static_cast<int>(in), 63, 64));
            }
        }
        if (lane == 0u)
        {
            out[0] = n ? mn : 0u; out[1] = mx; out[2] = p99; out[3] = total;
        }
    }

    __device__ void fluidStats(const double* __restrict__ partial, uint32_t nBlocks, double* __restrict__ out);

    __global__ void __launch_bounds__(kScanThreads) kStatsScan(StatsCounts c, const uint32_t* __restrict__ hist,
        const double* __restrict__ partial, uint32_t nBlocks, uint64_t* __restrict__ counts, double* __restrict__ fluid)
    {
        const uint32_t r = blockIdx.x;
        if (r < kRelations) { histogramStats(hist + static_cast<size_t>(r) * kHistBins, r < 3u ? c.nF : c.nR, counts + 4u * r); }
        else { fluidStats(partial, nBlocks, fluid); }
    }

    // per block of the scene's fluid: FP64 sums of the density error terms and of |v|, min and max |v|
    __global__ void __launch_bounds__(kBlock) kStatsFluid(const float4* __restrict__ vel, uint32_t off, uint32_t n,
        float rho0, double* __restrict__ partial)
    {
        __shared__ double red[4][kBlock / 64];
        __shared__ float vmin[kBlock / 64], vmax[kBlock / 64];
        const uint32_t q = blockIdx.x * kBlock + threadIdx.x;
        double raw = 0.0, pos = 0.0, ab = 0.0, vs = 0.0;
        float mn = 3.4e38f, mx = 0.0f;
        if (q < n)
        {
            const float4 v = vel[off + q];
            const float e = v.w / rho0 - 1.0f;
            raw = e; pos = e > 0.0f ? e : 0.0f; ab = __builtin_fabsf(e);
            const float m = __builtin_sqrtf(__builtin_fmaf(v.x, v.x, __builtin_fmaf(v.y, v.y, v.z * v.z)));
            vs = m; mn = m; mx = m;
        }
        for (int o = 32; o > 0; o >>= 1)
        {
            raw += __shfl_xor(raw, o, 64); pos += __shfl_xor(pos, o, 64);
            ab += __shfl_xor(ab, o, 64); vs += __shfl_xor(vs, o, 64);
            mn = fminf(mn, __shfl_xor(mn, o, 64)); mx = fmaxf(mx, __shfl_xor(mx, o, 64));
        }
        const uint32_t w = threadIdx.x >> 6;
        if ((threadIdx.x & 63u) == 0) { red[0][w] = raw; red[1][w] = pos; red[2][w] = ab; red[3][w] = vs; vmin[w] = mn; vmax[w] = mx; }
        __syncthreads();
        if (threadIdx.x == 0)
        {
            double a[4] = { 0, 0, 0, 0 };
            float lo = 3.4e38f, hi = 0.0f;
            for (uint32_t k = 0; k < kBlock / 64; k++)
            {
                for (int r = 0; r < 4; r++) { a[r] += red[r][k]; }
                lo = fminf(lo, vmin[k]); hi = fmaxf(hi, vmax[k]);
            }
            double* p = partial + 6ull * blockIdx.x;
            p[0] = a[0]; p[1] = a[1]; p[2] = a[2]; p[3] = a[3]; p[4] = lo; p[5] = hi;
        }
    }

    // the block partials summed in a fixed order: 1,024 threads stride over them, then a tree
    __device__ void fluidStats(const double* __restrict__ partial, uint32_t nBlocks, double* __restrict__ out)
    {
        __shared__ double red[6][kScanThreads / 64];
        double a[4] = { 0, 0, 0, 0 };
        double lo = 3.4e38, hi = 0.0;
        for (uint32_t b = threadIdx.x; b < nBlocks; b += kScanThreads)
        {
            for (int r = 0; r < 4; r++) { a[r] += partial[6ull * b + r]; }
            lo = fmin(lo, partial[6ull * b + 4]);
            hi = fmax(hi, partial[6ull * b + 5]);
        }
        for (int o = 32; o > 0; o >>= 1)
        {
            for (int r = 0; r < 4; r++) { a[r] += __shfl_xor(a[r], o, 64); }
            lo = fmin(lo, __shfl_xor(lo, o, 64));
            hi = fmax(hi, __shfl_xor(hi, o, 64));
        }
        const uint32_t w = threadIdx.x >> 6;
        if ((threadIdx.x & 63u) == 0u) { for (int r = 0; r < 4; r++) { red[r][w] = a[r]; } red[4][w] = lo; red[5][w] = hi; }
        __syncthreads();
        if (threadIdx.x != 0) { return; }
        for (uint32_t q = 1; q < kScanThreads / 64u; q++)
        {
            for (int r = 0; r < 4; r++) { a[r] += red[r][q]; }
            lo = fmin(lo, red[4][q]);
            hi = fmax(hi, red[5][q]);
        }
        for (int r = 0; r < 4; r++) { out[r] = a[r]; }
        out[4] = nBlocks ? lo : 0.0;
        out[5] = hi;
    }

    __global__ void __launch_bounds__(kBlock) kStatsClear(uint4* __restrict__ hist)
    {
        hist[blockIdx.x * kBlock + threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);
    }

    static inline uint32_t blocksN(uint64_t n) { return static_cast<uint32_t>((n + kBlock - 1) / kBlock); }

    // hist: kRelations x kHistBins words (cleared by a kernel, not a memset node, so the sequence can be
    // captured); partial: 6 doubles per block of nF; counts: per relation min, max, p99, sum; fluid: sums
    // of raw, positive, absolute error and |v|, min and max |v|
    void launchStats(hipStream_t s, const uint16_t* const (&c16)[3], const uint32_t* const (&c32)[3], uint32_t nF, uint32_t nR,
                     const float4* vel, uint32_t off, float rho0, uint32_t* hist, double* partial, uint64_t* counts, double* fluid)
    {
        StatsCounts c{ { c16[0], c16[1], c16[2] }, { c32[0], c32[1], c32[2] }, nF, nR };
        kStatsClear<<<kRelations * kHistBins / (4u * kBlock), kBlock, 0, s>>>(reinterpret_cast<uint4*>(hist));
        const uint32_t n = nF > nR ? nF : nR;
        if (n) { kStatsHist<<<min(256u, blocksN(n)), kBlock, 0, s>>>(c, hist); }
        if (nF) { kStatsFluid<<<blocksN(nF), kBlock, 0, s>>>(vel, off, nF, rho0, partial); }
        kStatsScan<<<kRelations + 1u, kScanThreads, 0, s>>>(c, hist, partial, blocksN(nF), counts, fluid);
    }

    // --- the statistics scratch of the allocation-free entry point (tsp_get_statistics_noalloc):
    //     one static array per GPU, for callers that cannot allocate device memory. Layout: the
    //     count histograms, the relations' (min, max, p99, sum), the fluid sums, then 6 FP64 block
    //     partials per 256 fluid particles of a scene of at most kStatsMaxFluid particles.
    //     Every call on one GPU shares that GPU's array: calls that overlap on one GPU (contexts
    //     on different streams) race, and each call leaves its values in it. ---
    constexpr uint32_t kStatsMaxFluid = 1u << 24;
    constexpr size_t kStatsHistOff = 0;
    constexpr size_t kStatsCountsOff = kStatsHistOff + sizeof(uint32_t) * kRelations * kHistBins;
    constexpr size_t kStatsFluidOff = kStatsCountsOff + 256;
    constexpr size_t kStatsPartialOff = kStatsFluidOff + 256;
    constexpr size_t kStatsScratchBytes = kStatsPartialOff + sizeof(double) * 6 * (kStatsMaxFluid / kBlock);
    static_assert(sizeof(uint64_t) * 24 <= 256 && sizeof(double) * 6 <= 256, "scratch layout");

    static __device__ __align__(256) unsigned char scratch[kStatsScratchBytes];

    constexpr int kStatsMaxDevices = 64;
    static void* scratchPtr[kStatsMaxDevices];
    static bool scratchReady[kStatsMaxDevices];
    static std::mutex scratchMutex;

    // once per device, with that device current: the device address of its copy of the array
    // (the array's name in host code is a host-side stand-in, not a device address)
    hipError_t statsScratchInit(int device)
    {
        if (device < 0 || device >= kStatsMaxDevices) { return hipErrorInvalidDevice; }
        std::lock_guard<std::mutex> lock(scratchMutex);
        if (scratchReady[device]) { return hipSuccess; }
        void* ptr = nullptr;
        const hipError_t rc = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (rc != hipSuccess) { return rc; }
        scratchPtr[device] = ptr;
        scratchReady[device] = true;
        return hipSuccess;
    }

    // the scratch buffers of one device (statsScratchInit ran for it), or false
    bool statsScratch(int device, uint32_t** hist, uint64_t** counts, double** fluid, double** partial,
                      uint32_t* maxFluid)
    {
        if (device < 0 || device >= kStatsMaxDevices) { return false; }
        std::lock_guard<std::mutex> lock(scratchMutex);
        if (!scratchReady[device]) { return false; }
        unsigned char* base = static_cast<unsigned char*>(scratchPtr[device]);
        *hist = reinterpret_cast<uint32_t*>(base + kStatsHistOff);
        *counts = reinterpret_cast<uint64_t*>(base + kStatsCountsOff);
        *fluid = reinterpret_cast<double*>(base + kStatsFluidOff);
        *partial = reinterpret_cast<double*>(base + kStatsPartialOff);
        *maxFluid = kStatsMaxFluid;
        return true;
    }
}
