// quotient_selftest.hip -- checks on the GPU that the quotient of the pair kernels as they run it
// (quotFrom with rootRcp's estimate of the reciprocal root, tsp_device.h) gives the same bits as the
// compiler's general correctly rounded root and quotient, over the whole range that the host allows
// (uploadConsts: 2^-60 <= |koutScale| <= 2^60 and no power of two, h >= 2^-30, 2h <= 2^31):
//   1. quotFrom(a, rootRcp(x)) over 2^33 pseudo-random pairs with |a| in [2^-60, 2^60] and sqrt(x) in
//      [2^-30, 2^31] (a tenth of them with mantissas at the ends of a binade);
//   2. the same over every mantissa of a and the 4,096 last floats x of a binade, for even and odd exponents:
//      the quotients that come closest to a midpoint have a root just below a power of two;
//   3. kgFactor<true> and kgShort with its correction against kgFactor<false> over every float d2 of the
//      outer branch, from h^2 to 4h^2, for h at the ends of the range and 48 pseudo-random h between, with
//      the constants that the host makes of them; a correction that does not fit in four bits keeps the
//      exact form, which may be no more than 8 of the floats of one h.
// Prints the counts and exits 0 when every case matches, 1 on a mismatch, 3 without a device.
#include <hip/hip_runtime.h>

#include <cmath>
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
        unsigned long long tested, bad, unfit, firstBad;
    };

    __host__ __device__ uint64_t mix64(uint64_t z)
    {
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return z ^ (z >> 31);
    }

    // a mantissa of 23 bits; one in ten lies within 8 of an end of its binade
    __device__ uint32_t mantissa(uint64_t z)
    {
        const uint32_t m = static_cast<uint32_t>(z) & 0x7fffffu;
        const uint32_t pick = static_cast<uint32_t>(z >> 32) % 20u;
        return pick == 0u ? m & 7u : (pick == 1u ? 0x7fffffu - (m & 7u) : m);
    }

    __global__ void __launch_bounds__(kThreads) kPairs(uint64_t n, uint64_t seed, Result* r)
    {
        const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
        unsigned long long tested = 0, bad = 0;
        for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        {
            const uint64_t z = mix64(seed + 0x9e3779b97f4a7c15ull * (i + 1)), u = mix64(z), v = mix64(u);
            const uint32_t ea = static_cast<uint32_t>(127 - 60 + (z % 120u));            // |a|: 2^-60 .. 2^60
            const uint32_t ex = static_cast<uint32_t>(127 - 60 + ((z >> 16) % 122u));    // x: 2^-60 .. 2^62
            const uint32_t ma = max(mantissa(u), 1u), mx = mantissa(v);
            const float a = __uint_as_float((static_cast<uint32_t>(z >> 63) << 31) | (ea << 23) | ma);
            const float x = __uint_as_float((ex << 23) | mx);
            float y;
            const float root = rootRcp(x, y);
            const float q = quotFrom(a, root, y);
            const float want = a / __builtin_sqrtf(x);
            tested++;
            if (__float_as_uint(q) != __float_as_uint(want) || __float_as_uint(root) != __float_as_uint(__builtin_sqrtf(x)))
            {
                bad++;
                atomicMin(&r->firstBad, static_cast<unsigned long long>(i));
            }
        }
        atomicAdd(&r->tested, tested);
        if (bad) { atomicAdd(&r->bad, bad); }
    }

    __global__ void __launch_bounds__(kThreads) kEnds(uint32_t exponent, uint32_t count, Result* r)
    {
        const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x, n = static_cast<uint64_t>(count) << 23;
        unsigned long long tested = 0, bad = 0;
        for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride)
        {
            const uint32_t ma = static_cast<uint32_t>(i) & 0x7fffffu;
            if (ma == 0u) { continue; }
            const float a = __uint_as_float((127u << 23) | ma);
            const float x = __uint_as_float((exponent << 23) | (0x7fffffu - static_cast<uint32_t>(i >> 23)));
            float y;
            const float root = rootRcp(x, y);
            tested++;
            if (__float_as_uint(quotFrom(a, root, y)) != __float_as_uint(a / __builtin_sqrtf(x)))
            {
                bad++;
                atomicMin(&r->firstBad, static_cast<unsigned long long>(i));
            }
        }
        atomicAdd(&r->tested, tested);
        if (bad) { atomicAdd(&r->bad, bad); }
    }

    __global__ void __launch_bounds__(kThreads) kOuter(Consts k, uint32_t lo, uint32_t n, Result* r)
    {
        const uint32_t stride = gridDim.x * blockDim.x;
        unsigned long long tested = 0, bad = 0, unfit = 0;
        for (uint64_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        {
            const uint32_t bits = lo + static_cast<uint32_t>(i);
            const float d2 = __uint_as_float(bits);
            const uint32_t exact = __float_as_uint(kgFactor<false>(d2, k));
            const uint32_t ulps = exact - __float_as_uint(kgShort(d2, k));
            const bool fits = ((ulps + 8u) & ~15u) == 0u;
            tested++;
            const bool wrong = __float_as_uint(kgFactor<true>(d2, k)) != exact
                               || (fits && __float_as_uint(addUlps(kgShort(d2, k), 0x1230u | (ulps & 15u))) != exact);
            if (!fits) { unfit++; }
            if (wrong) { bad++; atomicMin(&r->firstBad, static_cast<unsigned long long>(bits)); }
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
        z.firstBad = ~0ull;
        return check(hipMemcpy(dr, &z, sizeof(z), hipMemcpyHostToDevice), "H2D");
    }

    bool report(const char* name, Result* dr)
    {
        Result h{};
        if (!check(hipDeviceSynchronize(), name) || !check(hipMemcpy(&h, dr, sizeof(h), hipMemcpyDeviceToHost), "D2H")) { return false; }
        const bool ok = h.bad == 0 && h.tested > 0 && h.unfit <= 8;
        std::printf("%-48s tested %llu mismatches %llu unfit %llu%s\n", name, h.tested, h.bad, h.unfit, ok ? "" : " FAIL");
        if (h.bad) { std::printf("  first mismatch at input 0x%llx\n", h.firstBad); }
        std::fflush(stdout);
        return ok;
    }

    uint32_t bitsOf(float f)
    {
        uint32_t u;
        std::memcpy(&u, &f, 4);
        return u;
    }

    // the constants of a particle size as the host makes them, and whether it allows the short forms
    bool constsOf(float h, Consts& k)
    {
        const double hinv = 1.0 / static_cast<double>(h);
        k = Consts{};
        k.hinv = static_cast<float>(hinv);
        const float alpha = static_cast<float>(hinv * hinv * hinv / (4.0 * 3.14159265358979323846));
        k.ksize = 1.0f / k.hinv;
        k.ktwo = 2.0f / k.hinv;
        k.kinSlope = 9.0f * alpha * k.hinv * k.hinv * k.hinv;
        k.kinOff = -12.0f * alpha * k.hinv * k.hinv;
        k.koutScale = -3.0f * alpha * k.hinv * k.hinv * k.hinv;
        const float a = std::fabs(k.koutScale);
        int e;
        return a >= 0x1p-60f && a <= 0x1p60f && std::frexp(a, &e) != 0.5f && k.ksize >= 0x1p-30f && k.ktwo <= 0x1p31f;
    }
}

int main()
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) { std::fprintf(stderr, "no HIP device\n"); return 3; }
    Result* dr = nullptr;
    if (!check(hipMalloc(&dr, sizeof(Result)), "hipMalloc")) { return 1; }
    bool ok = reset(dr);
    kPairs<<<kBlocks, kThreads>>>(1ull << 33, 0x7469, dr);
    ok = report("a / sqrt(x), 2^33 random pairs in range", dr) && ok;
    for (const uint32_t exponent : { 127u, 128u })
    {
        ok = reset(dr) && ok;
        kEnds<<<kBlocks, kThreads>>>(exponent, 4096u, dr);
        ok = report(exponent == 127u ? "every a, x at the end of [1, 2)" : "every a, x at the end of [2, 4)", dr) && ok;
    }
    // the particle sizes that the gate lets through: |koutScale| = 3 / (4 pi h^6) within 2^-60 .. 2^60
    double lo = 1.0, hi = 1.0;
    Consts k;
    while (constsOf(static_cast<float>(lo / 1.0001), k)) { lo /= 1.0001; }
    while (constsOf(static_cast<float>(hi * 1.0001), k)) { hi *= 1.0001; }
    for (int q = 0; q < 50; q++)
    {
        const double u = q == 0 ? 0.0 : (q == 1 ? 1.0 : static_cast<double>(mix64(0x6871u + static_cast<uint64_t>(q)) >> 11) * 0x1p-53);
        const float h = static_cast<float>(lo * std::pow(hi / lo, u));
        if (!constsOf(h, k)) { continue; }
        char name[64];
        std::snprintf(name, sizeof(name), "gradient factor, h = %.9g", static_cast<double>(h));
        const float d2lo = (0.999f * k.ksize) * (0.999f * k.ksize), d2hi = k.ktwo * k.ktwo;
        ok = reset(dr) && ok;
        kOuter<<<kBlocks, kThreads>>>(k, bitsOf(d2lo), bitsOf(d2hi) - bitsOf(d2lo) + 1u, dr);
        ok = report(name, dr) && ok;
    }
    (void)hipFree(dr);
    std::printf("%s\n", ok ? "PASS" : "FAIL");
    return ok ? 0 : 1;
}
