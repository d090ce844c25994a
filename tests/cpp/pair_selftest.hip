// pair_selftest.hip -- checks on the GPU that the short forms of the pair kernels (tsp_device.h)
// give the same bits as the general correctly rounded lowering:
//   1. rootRcp over 0 and every finite float from 2^-96 up (its domain);
//   2. kgFactor<true> against kgFactor<false> over d2 = 0 and every float from (h / 128)^2 to r^2,
//      for particle sizes h from 0.0008 to 1;
//   3. over the same d2: kgShort moved by the four-bit correction that kSourceDiag would store is
//      kgFactor<false>, except where the correction does not fit (sqrt(d2) rounded above 2h: the
//      block then keeps the exact form), which may be no more than 8 of the floats of one h.
// Prints the counts and exits 0 when every case matches, 1 on a mismatch, 3 without a device.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstring>

#include "tsp_device.h"

using namespace tsp;

namespace
{
    constexpr int kThreads = 256;
    constexpr int kBlocks = 4096;

    struct Result
    {
        unsigned long long tested, bad, unfit;
        uint32_t firstBad, pad;
    };

    __global__ void __launch_bounds__(kThreads) kRoots(uint32_t lo, uint32_t n, Result* r)
    {
        unsigned long long tested = 0, bad = 0;
        for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i <= n; i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
        {
            const uint32_t bits = i == n ? 0u : lo + static_cast<uint32_t>(i);
            float y;
            const float x = __uint_as_float(bits);
            const float a = rootRcp(x, y), b = __builtin_sqrtf(x);
            tested++;
            if (__float_as_uint(a) != __float_as_uint(b)) { bad++; atomicMin(&r->firstBad, bits); }
        }
        atomicAdd(&r->tested, tested);
        if (bad) { atomicAdd(&r->bad, bad); }
    }

    __global__ void __launch_bounds__(kThreads) kFactors(Consts k, uint32_t lo, uint32_t n, Result* r)
    {
        unsigned long long tested = 0, bad = 0, unfit = 0;
        for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i <= n; i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
        {
            const uint32_t bits = i == n ? 0u : lo + static_cast<uint32_t>(i);
            const float d2 = __uint_as_float(bits);
            const uint32_t exact = __float_as_uint(kgFactor<false>(d2, k));
            const uint32_t ulps = exact - __float_as_uint(kgShort(d2, k));
            const bool fits = ((ulps + 8u) & ~15u) == 0u;
            const uint32_t entry = 0x1230u | (ulps & 15u);
            tested++;
            const bool wrong = __float_as_uint(kgFactor<true>(d2, k)) != exact
                               || (fits && __float_as_uint(addUlps(kgShort(d2, k), entry)) != exact);
            if (!fits) { unfit++; }
            if (wrong) { bad++; atomicMin(&r->firstBad, bits); }
        }
        atomicAdd(&r->tested, tested);
        if (bad) { atomicAdd(&r->bad, bad); }
        if (unfit) { atomicAdd(&r->unfit, unfit); }
    }

    bool check(hipError_t e, const char* what)
    {
        if (e != hipSuccess) { std::fprintf(stderr, "%s: %s\n", what, hipGetErrorString(e)); return false; }
        return true;
    }

    bool reset(Result* dr)
    {
        Result z{};
        z.firstBad = 0xffffffffu;
        return check(hipMemcpy(dr, &z, sizeof(z), hipMemcpyHostToDevice), "H2D");
    }

    bool report(const char* name, Result* dr)
    {
        Result h{};
        if (!check(hipDeviceSynchronize(), name) || !check(hipMemcpy(&h, dr, sizeof(h), hipMemcpyDeviceToHost), "D2H")) { return false; }
        const bool ok = h.bad == 0 && h.tested > 0 && h.unfit <= 8;
        std::printf("%-40s tested %llu mismatches %llu unfit %llu%s\n", name, h.tested, h.bad, h.unfit, ok ? "" : " FAIL");
        if (h.bad) { std::printf("  first mismatch at input 0x%08x\n", h.firstBad); }
        std::fflush(stdout);
        return ok;
    }

    uint32_t bitsOf(float f)
    {
        uint32_t u;
        std::memcpy(&u, &f, 4);
        return u;
    }
}

int main()
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) { std::fprintf(stderr, "no HIP device\n"); return 3; }
    Result* dr = nullptr;
    if (!check(hipMalloc(&dr, sizeof(Result)), "hipMalloc")) { return 1; }
    bool ok = reset(dr);
    kRoots<<<kBlocks, kThreads>>>(0x0f800000u, 0x7f800000u - 0x0f800000u, dr);
    ok = report("rootRcp, 0 and every float in [2^-96, inf)", dr) && ok;
    for (const float h : { 0.0008f, 0.001f, 0.002f, 0.004f, 0.005f, 0.00754717f, 0.01f, 0.02f, 0.05f, 0.1f, 0.5f, 1.0f })
    {
        // the kernel constants as the host computes them
        Consts k{};
        const double hinv = 1.0 / static_cast<double>(h);
        k.hinv = static_cast<float>(hinv);
        const float alpha = static_cast<float>(hinv * hinv * hinv / (4.0 * 3.14159265358979323846));
        k.ksize = 1.0f / k.hinv;
        k.ktwo = 2.0f / k.hinv;
        k.kinSlope = 9.0f * alpha * k.hinv * k.hinv * k.hinv;
        k.kinOff = -12.0f * alpha * k.hinv * k.hinv;
        k.koutScale = -3.0f * alpha * k.hinv * k.hinv * k.hinv;
        const float r = 2.0f * h, lo = (h / 128.0f) * (h / 128.0f);
        char name[64];
        std::snprintf(name, sizeof(name), "gradient factor, h = %g", static_cast<double>(h));
        ok = reset(dr) && ok;
        kFactors<<<kBlocks, kThreads>>>(k, bitsOf(lo), bitsOf(r * r) - bitsOf(lo) + 1u, dr);
        ok = report(name, dr) && ok;
    }
    (void)hipFree(dr);
    std::printf("%s\n", ok ? "PASS" : "FAIL");
    return ok ? 0 : 1;
}
