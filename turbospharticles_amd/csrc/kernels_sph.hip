// kernels_sph.hip -- IISPH solver kernels of the step on gfx950.
//
// One thread per fluid particle; a wave64 reads one SELL slice, so the list loads of a neighbor
// column are one row. Every kernel first issues the loads that depend on nothing but the block (list
// heads, slice headers, first entries, halo indices), then the ones that depend on those (the halo
// records, the particle's own), and only then waits: a block starts its sums after two memory
// latencies instead of eight, which also shortens the first and the last blocks of a large launch.
// Headers, constants and scene records are scalar loads (uniformLoad). Measured against the loads in
// order of use: 1M cube drop kJacobi 47.4 to 39.3 us, kPressureAcc 38.0 to 31.0, kDensity 36.3 to
// 32.7, kSourceDiag 69.8 to 59.8, kNonPressure 64.2 to 62.0; 64k particles kPressureAcc 12.8 to 11.0,
// kJacobi 12.4 to 10.4. FF sums use the reference CPU's dict-chunk
// form (one scale after the sum), FB/FR sums its normal form, each in the list order the fill
// wrote (CPU/backend/sph_solver.cpp):
//   kDensity         Density_ChunkedSELL                            :734-890
//   kNonPressure     NonPressureAcceleration_ChunkedSELL            :892-1149
//   kSourceDiag      SourceTermAndDiagonalElementAndPressureJacobiInit :1225-1504
//   kPressureAcc     PressureAcceleration_ChunkedSELL               :1507-1715
//   kJacobi          PressureRelaxedJacobiSolver_ChunkedSELL        :1781-2049, FP64 error partials
//   finalizeSweep    the error sums, averages and TerminationConditionSatisfied (:205-261, :686-732)
//                    decided on the device by block 0 of the next sweep's kPressureAcc (kFinalize
//                    after the last sweep of a group), so no host round trip is needed per sweep
//   kIntegration     Integration                                    :2051-2089
// Rigid coupling (CPU/backend/cpu_backend.cpp:2001-2303, sph_solver.cpp:1151-1223, :1717-1778):
// particle kinematics, reaction forces over the RF lists, FP64 per-body force/torque sums,
// prediction and semi-implicit integration with Gram-Schmidt re-orthonormalization.
#include "tsp_device.h"

namespace tsp
{
    // two records of a halo neighbor
    struct Pair4
    {
        float4 a, b;
    };

    struct BoundaryRec
    {
        float4 p;
        float vol;
    };

    template <bool kFast>
    __global__ void __launch_bounds__(kBlock) kDensity(Dev d)
    {
        if (stopped(d)) { return; }
        __shared__ float4 hp[kHaloMax];
        const uint32_t blk = xcdBlock();
        const Lists l = listsAt(d, blk);
        const SlotList slots = slotsOf(d, l);
        const Halo h = haloOf(d, blk);
        const uint32_t sc = uniformLoad(&d.blockScene[blk]);
        const Consts k = uniformLoad(&d.consts[sc]);
        const Scene S = uniformLoad(&d.scenes[sc]);
        const uint32_t i = l.i;
        const float4 pi = d.pos[i];
        stageHalo(h, [&](uint32_t j) { return d.pos[j]; }, [&](uint32_t q, const float4& r) { hp[q] = r; });
        __syncthreads();
        if (i - S.offF >= S.nF) { return; }
        const float xi = pi.x, yi = pi.y, zi = pi.z;
        float dF;
        const auto sumFF = [&](auto&& ffTerm)
        {
            if (h.any) { visitSlots(slots, [&](uint32_t q, uint32_t) { ffTerm(recAt(hp, q)); }); }
            else { visit(l.list(d, REL_FF), [&](uint32_t j) { ffTerm(d.pos[j]); }); }
        };
        if (slots.n <= kDictMax)
        {
            // dict chunk: unscaled weights, scaled once (sph_solver.cpp:797-810)
            float wsum = 0.0f;
            sumFF([&](const float4& pj) { wsum += kwUnscaled<kFast>(dist2(xi - pj.x, yi - pj.y, zi - pj.z), k); });
            dF = wsum * k.weightScale;
        }
        else
        {
            // normal chunk: the alpha-scaled weight per neighbor (sph_solver.cpp:826-831)
            float s = 0.0f;
            sumFF([&](const float4& pj) { s = __builtin_fmaf(k.mass, kwNormal<kFast>(xi - pj.x, yi - pj.y, zi - pj.z, k), s); });
            dF = s;
        }
        float dB = 0.0f, dR = 0.0f;
        visitGather(d, l, REL_FB, [&](uint32_t j) { return d.bpos[j]; }, [&](const float4& bj)
        {
            dB = __builtin_fmaf(bj.w, kwNormal<kFast>(xi - bj.x, yi - bj.y, zi - bj.z, k), dB);
        });
        visit(l.list(d, REL_FR), [&](uint32_t j)
        {
            const float4 rj = d.rpos[j];
            dR = __builtin_fmaf(rj.w, kwNormal(xi - rj.x, yi - rj.y, zi - rj.z, k), dR);
        });
        d.vel[i].w = dF + dB + dR;
    }

    template <bool kFast>
    __global__ void __launch_bounds__(kBlock) kNonPressure(Dev d)
    {
        if (stopped(d)) { return; }
        __shared__ float4 hp[kHaloMax], hv[kHaloMax];
        const uint32_t blk = xcdBlock();
        const Lists l = listsAt(d, blk);
        const SlotList slots = slotsOf(d, l);
        const Halo h = haloOf(d, blk);
        const uint32_t sc = uniformLoad(&d.blockScene[blk]);
        const Consts k = uniformLoad(&d.consts[sc]);
        const Scene S = uniformLoad(&d.scenes[sc]);
        const uint32_t i = l.i;
        const float4 pi = d.pos[i], vi = d.vel[i];
        stageHalo(h, [&](uint32_t j) { return Pair4{ d.pos[j], d.vel[j] }; }, [&](uint32_t q, const Pair4& r) { hp[q] = r.a; hv[q] = r.b; });
        __syncthreads();
        if (i - S.offF >= S.nF) { return; }
        const float xi = pi.x, yi = pi.y, zi = pi.z, vxi = vi.x, vyi = vi.y, vzi = vi.z;
        float aFx = 0.0f, aFy = 0.0f, aFz = 0.0f;
        // dict chunks scale by the mass after the sum, normal chunks per neighbor (sph_solver.cpp:974-1049)
        const bool dict = slots.n <= kDictMax;
        // the two forms as two loops (a wave runs the normal one only for a list longer than kDictMax)
        const auto sumFF = [&](auto dictFlag)
        {
            constexpr bool kDict = decltype(dictFlag)::value;
            const auto ffTerm = [&](const float4& pj, const float4& vj)
            {
                const float dx = xi - pj.x, dy = yi - pj.y, dz = zi - pj.z;
                const float dvx = vxi - vj.x, dvy = vyi - vj.y, dvz = vzi - vj.z;
                const float d2 = dist2(dx, dy, dz);
                const float kg = kgFactor<kFast>(d2, k);
                const float dot = __builtin_fmaf(dvx, dx, __builtin_fmaf(dvy, dy, dvz * dz));
                const float rj = vmax(vj.w, 1e-7f);
                const float coeff = (kDict ? dot : k.mass * dot) / (rj * (d2 + k.hsqEps)) * kg;
                aFx = __builtin_fmaf(coeff, dx, aFx);
                aFy = __builtin_fmaf(coeff, dy, aFy);
                aFz = __builtin_fmaf(coeff, dz, aFz);
            };
            if (h.any) { visitSlots(slots, [&](uint32_t q, uint32_t) { ffTerm(recAt(hp, q), recAt(hv, q)); }); }
            else { visit(l.list(d, REL_FF), [&](uint32_t j) { ffTerm(d.pos[j], d.vel[j]); }); }
        };
        if (dict) { sumFF(Flag<true>{}); } else { sumFF(Flag<false>{}); }
        if (dict) { aFx *= k.mass; aFy *= k.mass; aFz *= k.mass; }
        float aBx = 0.0f, aBy = 0.0f, aBz = 0.0f;
        visitGather(d, l, REL_FB, [&](uint32_t j) { return BoundaryRec{ d.bpos[j], d.bvol[j] }; }, [&](const BoundaryRec& r)
        {
            const float4& bj = r.p;
            const float dx = xi - bj.x, dy = yi - bj.y, dz = zi - bj.z;
            const float d2 = dist2(dx, dy, dz);
            const float f = kgFactor<kFast>(d2, k);
            const float gx = f * dx, gy = f * dy, gz = f * dz;
            const float dvx = vxi - 0.0f, dvy = vyi - 0.0f, dvz = vzi - 0.0f;
            const float dot = __builtin_fmaf(dvx, dx, __builtin_fmaf(dvy, dy, dvz * dz));
            const float coeff = (r.vol * dot) / (d2 + k.hsqEps);
            aBx = __builtin_fmaf(coeff, gx, aBx);
            aBy = __builtin_fmaf(coeff, gy, aBy);
            aBz = __builtin_fmaf(coeff, gz, aBz);
        });
        float aRx = 0.0f, aRy = 0.0f, aRz = 0.0f;
        visit(l.list(d, REL_FR), [&](uint32_t j)
        {
            const float4 rj = d.rpos[j], uj = d.rvel[j];
            const float dx = xi - rj.x, dy = yi - rj.y, dz = zi - rj.z;
            const float d2 = dist2(dx, dy, dz);
            const float f = kgFactor(d2, k);
            const float gx = f * dx, gy = f * dy, gz = f * dz;
            const float dvx = vxi - uj.x, dvy = vyi - uj.y, dvz = vzi - uj.z;
            const float dot = __builtin_fmaf(dvx, dx, __builtin_fmaf(dvy, dy, dvz * dz));
            const float coeff = (uj.w * dot) / (d2 + k.hsqEps);
            aRx = __builtin_fmaf(coeff, gx, aRx);
            aRy = __builtin_fmaf(coeff, gy, aRy);
            aRz = __builtin_fmaf(coeff, gz, aRz);
        });
        const float ax = aFx * k.visF + (aBx + aRx) * k.visB + k.gx;
        const float ay = aFy * k.visF + (aBy + aRy) * k.visB + k.gy;
        const float az = aFz * k.visF + (aBz + aRz) * k.visB + k.gz;
        d.vp[i] = make_float4(__builtin_fmaf(ax, k.dt, vxi), __builtin_fmaf(ay, k.dt, vyi), __builtin_fmaf(az, k.dt, vzi), 0.0f);
    }

    // TerminationConditionSatisfied, sph_solver.cpp:686-732
    __device__ __forceinline__ bool terminated(const Solve& s, const Consts& k)
    {
        if (s.iters < k.minIters) { return false; }
        if (s.iters >= k.maxIters) { return true; }
        switch (k.termCond)
        {
        case 0: return s.iters >= k.fixedIters;
        case 1: return s.avgRaw <= k.densityDevTarget;
        case 2: return s.avgPos <= k.densityDevTarget;
        case 3: return s.avgAbs <= k.densityDevTarget;
        default: return s.iters >= 3;
        }
    }

    // the solver state before the first sweep: N_solverIters_ = 1, errors 0, then the
    // increment and error decision of the first sweep (sph_solver.cpp:207-235); by one block
    __device__ __forceinline__ void solverInit(const Dev& d)
    {
        for (uint32_t sc = threadIdx.x; sc < d.nScenes; sc += kBlock)
        {
            Solve& s = d.solve[sc];
            const Consts& k = d.consts[sc];
            const bool any = d.scenes[sc].nF > 0;
            s.iters = any ? 1u : 0u;
            s.avgRaw = s.avgPos = s.avgAbs = 0.0f;
            s.sumRaw = s.sumPos = s.sumAbs = 0.0;
            s.converged = any ? 0u : 1u;
            s.sweeps = 0;
            s.pending = 0;
            s.iters++;
            s.compute = (s.iters >= k.minIters && (k.termCond != 0 || terminated(s, k))) ? 1u : 0u;
            for (uint32_t q = 0; q < kBarWords; q += kBarLine) { d.solveBar[static_cast<size_t>(sc) * kBarWords + q] = 0u; }
        }
        for (uint32_t q = threadIdx.x; q < kFlagCopies * kSolveBlocksMost; q += kBlock) { d.solveFlag[q] = 0u; }
    }

    template <bool kFast>
    __global__ void __launch_bounds__(kBlock) kSourceDiag(Dev d)
    {
        if (stopped(d)) { return; }
        // the block after the tiles' readies the solver states
        const uint32_t nTiles = d.nF / kBlock;
        if (blockIdx.x == nTiles) { solverInit(d); return; }
        __shared__ float4 hp[kHaloMax], hv[kHaloMax];
        const uint32_t blk = xcdBlock(nTiles);
        const Lists l = listsAt(d, blk);
        const SlotList slots = slotsOf(d, l);
        const Halo h = haloOf<false>(d, blk);   // (this kernel writes ulps)
        const uint32_t sc = uniformLoad(&d.blockScene[blk]);
        const Consts k = uniformLoad(&d.consts[sc]);
        const Scene S = uniformLoad(&d.scenes[sc]);
        const uint32_t i = l.i;
        const float4 pi = d.pos[i], vi = d.vp[i];
        const float rho = d.vel[i].w;
        stageHalo(h, [&](uint32_t j) { return Pair4{ d.pos[j], d.vp[j] }; }, [&](uint32_t q, const Pair4& r) { hp[q] = r.a; hv[q] = r.b; });
        __syncthreads();
        if (i - S.offF >= S.nF) { return; }
        const float xi = pi.x, yi = pi.y, zi = pi.z, vxi = vi.x, vyi = vi.y, vzi = vi.z;
        float sF = 0.0f, cFx = 0.0f, cFy = 0.0f, cFz = 0.0f, g2 = 0.0f;
        const auto ffSum = [&](float dx, float dy, float dz, float d2, float kg, const float4& vj)
        {
            const float dvx = vxi - vj.x, dvy = vyi - vj.y, dvz = vzi - vj.z;
            const float st = __builtin_fmaf(dvx, dx, __builtin_fmaf(dvy, dy, dvz * dz));
            sF = __builtin_fmaf(kg, st, sF);
            cFx = __builtin_fmaf(kg, dx, cFx);
            cFy = __builtin_fmaf(kg, dy, cFy);
            cFz = __builtin_fmaf(kg, dz, cFz);
            g2 = __builtin_fmaf(kg, kg * d2, g2);
        };
        uint32_t far = 0;   // a correction of this list does not fit its four bits
        if (h.any)
        {
            visitSlots(slots, [&](uint32_t q, uint32_t row)
            {
                const float4& pj = recAt(hp, q);
                const float dx = xi - pj.x, dy = yi - pj.y, dz = zi - pj.z;
                const float d2 = dist2(dx, dy, dz);
                const float kg = kgFactor<kFast>(d2, k);
                if (kFast)
                {
                    // the pair's kgShort correction for this step's sweeps
                    const uint32_t ulps = static_cast<uint32_t>(__float_as_int(kg) - __float_as_int(kgShort(d2, k)));
                    far |= (ulps + 8u) & ~15u;
                    slots.p[row * kSlice] = static_cast<uint16_t>(q | (ulps & 15u));
                }
                ffSum(dx, dy, dz, d2, kg, recAt(hv, q));
            });
        }
        else
        {
            visit(l.list(d, REL_FF), [&](uint32_t j)
            {
                const float4 pj = d.pos[j];
                const float dx = xi - pj.x, dy = yi - pj.y, dz = zi - pj.z;
                const float d2 = dist2(dx, dy, dz);
                ffSum(dx, dy, dz, d2, kgFactor<kFast>(d2, k), d.vp[j]);
            });
        }
        if (far) { d.haloInfo[blk].ulps = 0u; }
        float sB = 0.0f, cBx = 0.0f, cBy = 0.0f, cBz = 0.0f;
        visitGather(d, l, REL_FB, [&](uint32_t j) { return d.bpos[j]; }, [&](const float4& bj)
        {
            const float dx = xi - bj.x, dy = yi - bj.y, dz = zi - bj.z;
            const float f = kgFactor<kFast>(dist2(dx, dy, dz), k);
            const float gx = f * dx, gy = f * dy, gz = f * dz;
            const float dvx = vxi - 0.0f, dvy = vyi - 0.0f, dvz = vzi - 0.0f;
            const float st = __builtin_fmaf(dvx, gx, __builtin_fmaf(dvy, gy, dvz * gz));
            const float psi = bj.w;
            sB = __builtin_fmaf(psi, st, sB);
            cBx = __builtin_fmaf(psi, gx, cBx);
            cBy = __builtin_fmaf(psi, gy, cBy);
            cBz = __builtin_fmaf(psi, gz, cBz);
        });
        float sR = 0.0f, cRx = 0.0f, cRy = 0.0f, cRz = 0.0f;
        visit(l.list(d, REL_FR), [&](uint32_t j)
        {
            const float4 rj = d.rpos[j], uj = d.rvp[j];
            const float dx = xi - rj.x, dy = yi - rj.y, dz = zi - rj.z;
            const float f = kgFactor(dist2(dx, dy, dz), k);
            const float gx = f * dx, gy = f * dy, gz = f * dz;
            const float dvx = vxi - uj.x, dvy = vyi - uj.y, dvz = vzi - uj.z;
            const float st = __builtin_fmaf(dvx, gx, __builtin_fmaf(dvy, gy, dvz * gz));
            const float psi = rj.w;
            sR = __builtin_fmaf(psi, st, sR);
            cRx = __builtin_fmaf(psi, gx, cRx);
            cRy = __builtin_fmaf(psi, gy, cRy);
            cRz = __builtin_fmaf(psi, gz, cRz);
        });
        sF *= k.mass;
        const float src = k.rho0 - rho - k.dt * (sF + sB + sR);
        const float ctx = cFx * k.cFacF + (cBx + cRx) * k.cFacB;
        const float cty = cFy * k.cFacF + (cBy + cRy) * k.cFacB;
        const float ctz = cFz * k.cFacF + (cBz + cRz) * k.cFacB;
        const float dA = k.mass * __builtin_fmaf(ctx, cFx, __builtin_fmaf(cty, cFy, ctz * cFz));
        const float dB = k.mass * k.dFacB * g2;
        const float dC = __builtin_fmaf(ctx, cBx + cRx, __builtin_fmaf(cty, cBy + cRy, ctz * (cBz + cRz)));
        const float diag = k.dtsq * (dA + dB + dC);
        const bool valid = __builtin_fabsf(diag) > 1e-7f;
        const float cold = k.omega * (src / diag);
        float init = cold;
        if (k.warm > 0.0f)
        {
            const float prev = pi.w;
            init = prev > 0.0f ? k.warm * prev : cold;
        }
        d.source[i] = src;
        d.diag[i] = diag;
        d.pos[i].w = vmax(0.0f, valid ? init : 0.0f);
    }

    // the value of the lane `kRot` further in the lane's row of 16 (rotating)
    template <int kRot>
    __device__ __forceinline__ double rowRotate(double v)
    {
        const long long u = __double_as_longlong(v);
        const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u), 0x120 + kRot, 0xf, 0xf, true);
        const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), 0x120 + kRot, 0xf, 0xf, true);
        return __longlong_as_double(static_cast<long long>(hi) << 32 | static_cast<uint32_t>(lo));
    }

    // sum over the 64 lanes of a wave (a fixed xor tree: the same order on every run). After the steps of
    // 32, 16 and 8 lanes a row repeats every 8 lanes, so a rotation by 4 pairs the lanes that an xor of 4
    // pairs, and so on.
    __device__ __forceinline__ double waveSum(double v)
    {
        v += __shfl_xor(v, 32, 64);
        v += __shfl_xor(v, 16, 64);
        v += rowRotate<8>(v);
        v += rowRotate<4>(v);
        v += rowRotate<2>(v);
        v += rowRotate<1>(v);
        return v;
    }

    // threads of a solver sweep block (one 256-particle tile per block)
    constexpr uint32_t kSweepThreads = kBlock;

    // the bookkeeping of one scene after a Jacobi sweep (sph_solver.cpp:207-261): the scene's block
    // partials summed in a fixed order, the averages, TerminationConditionSatisfied and the error
    // decision of the next sweep. Run by one whole block of kSweepThreads; nTot is the grid size of
    // the sweep.
    __device__ void finalizeSweep(const Dev& d, uint32_t sc, uint32_t nTot)
    {
        __shared__ double red[3][kSweepThreads / 64];
        __shared__ uint32_t flags[2];
        Solve& s = d.solve[sc];
        const Consts& k = d.consts[sc];
        const uint32_t b0 = d.scenes[sc].blk0, nBlocks = d.scenes[sc].nBlk;
        // one read of the flags for the whole block, so every wave takes the same path (the first
        // barrier lets a previous call's readers finish before thread 0 writes them again)
        __syncthreads();
        if (threadIdx.x == 0) { flags[0] = s.pending; flags[1] = s.compute; }
        __syncthreads();
        if (!flags[0]) { return; }
        const bool compute = flags[1] != 0u;
        if (compute)
        {
            for (int r = 0; r < 3; r++)
            {
                const double* src = d.errPartial + static_cast<size_t>(r) * nTot + b0;
                double a = 0.0;
                uint32_t b = threadIdx.x;
                constexpr uint32_t kT = kSweepThreads;
                for (; b + 3 * kT < nBlocks; b += 4 * kT)
                {
                    const double v0 = src[b], v1 = src[b + kT], v2 = src[b + 2 * kT], v3 = src[b + 3 * kT];
                    a += v0; a += v1; a += v2; a += v3;
                }
                for (; b < nBlocks; b += kT) { a += src[b]; }
                a = waveSum(a);
                if ((threadIdx.x & 63u) == 0) { red[r][threadIdx.x >> 6] = a; }
            }
            __syncthreads();
            if (threadIdx.x == 0)
            {
                for (int r = 0; r < 3; r++)
                {
                    double a = red[r][0];
                    for (uint32_t w = 1; w < kSweepThreads / 64; w++) { a += red[r][w]; }
                    red[r][0] = a;
                }
            }
        }
        if (threadIdx.x == 0)
        {
            s.pending = 0;
            s.sweeps++;
            if (compute)
            {
                s.sumRaw = red[0][0]; s.sumPos = red[1][0]; s.sumAbs = red[2][0];
                const float n = static_cast<float>(d.scenes[sc].nF);
                s.avgRaw = static_cast<float>(red[0][0]) / n;
                s.avgPos = static_cast<float>(red[1][0]) / n;
                s.avgAbs = static_cast<float>(red[2][0]) / n;
            }
            if (terminated(s, k))
            {
                s.converged = 1u;
            }
            else
            {
                s.iters++;
                s.compute = (s.iters >= k.minIters && (k.termCond != 0 || terminated(s, k))) ? 1u : 0u;
            }
        }
        __syncthreads();
    }

    // the FR terms of a pressure acceleration
    __device__ __forceinline__ void pressureFR(const Dev& d, const Lists& l, const Consts& k, const float4& p4, float& ax, float& ay, float& az)
    {
        visit(l.list(d, REL_FR), [&](uint32_t j)
        {
            const float4 rj = d.rpos[j];
            const float dx = p4.x - rj.x, dy = p4.y - rj.y, dz = p4.z - rj.z;
            const float f = kgFactor(dist2(dx, dy, dz), k);
            const float coeff = k.presOuterB * rj.w * p4.w;
            ax = __builtin_fmaf(coeff, f * dx, ax);
            ay = __builtin_fmaf(coeff, f * dy, ay);
            az = __builtin_fmaf(coeff, f * dz, az);
        });
    }

    // the pressure acceleration of a particle at p4 (x, y, z, pressure): its FF sum over the staged halo, or
    // over posOf(j) in a block without one, and its FB and FR sums
    template <bool kFast, typename PosOf>
    __device__ __forceinline__ void pressureAt(const Dev& d, const Lists& l, const SlotList& slots, const Halo& h, const float4* hp,
        const Consts& k, const float4& p4, PosOf&& posOf, float (&a)[3])
    {
        const float xi = p4.x, yi = p4.y, zi = p4.z, pi = p4.w;
        float sx = 0.0f, sy = 0.0f, sz = 0.0f;
        // dict chunks sum (p_i + p_j) kg and scale once; normal chunks scale each neighbor's
        // pressure term (sph_solver.cpp:1573-1640)
        const bool dict = slots.n <= kDictMax;
        const float outerF = k.mass * pi * k.presDis;
        // the two forms as two loops (a wave runs the normal one only for a list longer than kDictMax)
        const auto sumFF = [&](auto dictFlag)
        {
            constexpr bool kDict = decltype(dictFlag)::value;
            // q: the pair's halo entry where its low bits correct kgShort (kShort)
            const auto ffTerm = [&](const float4& pj, uint32_t q, auto shortFlag)
            {
                constexpr bool kShort = decltype(shortFlag)::value;
                const float dx = xi - pj.x, dy = yi - pj.y, dz = zi - pj.z;
                const float d2 = dist2(dx, dy, dz);
                const float kg = kShort ? addUlps(kgShort(d2, k), q) : kgFactor<kFast>(d2, k);
                const float coeff = (kDict ? pi + pj.w : outerF + k.mass * pj.w * k.presDis) * kg;
                sx = __builtin_fmaf(coeff, dx, sx);
                sy = __builtin_fmaf(coeff, dy, sy);
                sz = __builtin_fmaf(coeff, dz, sz);
            };
            if (kFast && h.ulps) { visitSlots(slots, [&](uint32_t q, uint32_t) { ffTerm(recAt(hp, q & kSlotMask), q, Flag<true>{}); }); }
            else if (h.any) { visitSlots(slots, [&](uint32_t q, uint32_t) { ffTerm(recAt(hp, q & kSlotMask), q, Flag<false>{}); }); }
            else { visit(l.list(d, REL_FF), [&](uint32_t j) { ffTerm(posOf(j), 0u, Flag<false>{}); }); }
        };
        if (dict) { sumFF(Flag<true>{}); } else { sumFF(Flag<false>{}); }
        float ax = dict ? sx * k.presOuterFF : sx, ay = dict ? sy * k.presOuterFF : sy, az = dict ? sz * k.presOuterFF : sz;
        visitGather(d, l, REL_FB, [&](uint32_t j) { return d.bpos[j]; }, [&](const float4& bj)
        {
            const float dx = xi - bj.x, dy = yi - bj.y, dz = zi - bj.z;
            const float f = kgFactor<kFast>(dist2(dx, dy, dz), k);
            const float coeff = k.presOuterB * bj.w * pi;
            ax = __builtin_fmaf(coeff, f * dx, ax);
            ay = __builtin_fmaf(coeff, f * dy, ay);
            az = __builtin_fmaf(coeff, f * dz, az);
        });
        pressureFR(d, l, k, p4, ax, ay, az);
        a[0] = 0.0f - ax; a[1] = 0.0f - ay; a[2] = 0.0f - az;
    }

    // one tile of a sweep's pressure accelerations. Blocks that see the solve converged skip their
    // particles: the final launch (sweep = false) recomputes every a^p.
    template <bool kFast>
    __device__ __forceinline__ void pressureAccTile(const Dev& d, uint32_t blk, bool sweep)
    {
        __shared__ float4 hp[kHaloMax];
        __shared__ uint32_t skip;
        const Lists l = listsAt(d, blk);
        const SlotList slots = slotsOf(d, l);
        const Halo h = haloOf(d, blk);
        const uint32_t sc = uniformLoad(&d.blockScene[blk]);
        const Consts k = uniformLoad(&d.consts[sc]);
        const Scene S = uniformLoad(&d.scenes[sc]);
        if (sweep)
        {
            // one read per block, so the whole block leaves together
            if (threadIdx.x == 0) { skip = __hip_atomic_load(&d.solve[sc].converged, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
            __syncthreads();
            if (skip) { return; }
        }
        const uint32_t i = l.i;
        const float4 p4 = d.pos[i];
        stageHalo(h, [&](uint32_t j) { return d.pos[j]; }, [&](uint32_t q, const float4& r) { hp[q] = r; });
        __syncthreads();
        if (i - S.offF >= S.nF) { return; }
        float a[3];
        pressureAt<kFast>(d, l, slots, h, hp, k, p4, [&](uint32_t j) { return d.pos[j]; }, a);
        d.ap[i] = make_float4(a[0], a[1], a[2], 0.0f);
    }

    template <bool kFast>
    __global__ void __launch_bounds__(kSweepThreads) TSP_WAVES_ATTR(TSP_TUNE_PA_WAVES) kPressureAcc(Dev d, bool sweep, uint32_t nTiles)
    {
        if (stopped(d)) { return; }
        // a sweep launch first finishes the bookkeeping of the previous Jacobi sweep, which the next Jacobi
        // launch reads: block b that of scenes b, b + grid, ...
        if (sweep)
        {
            for (uint32_t q = blockIdx.x; q < d.nScenes; q += gridDim.x) { finalizeSweep(d, q, nTiles); }
        }
        pressureAccTile<kFast>(d, xcdBlock(), sweep);
    }

    __device__ __forceinline__ void addError(float pred, const Consts& k, double& eRaw, double& ePos, double& eAbs)
    {
        const double e = static_cast<double>(pred / k.rho0);
        eRaw += e;
        ePos += 0.0 < e ? e : 0.0;
        eAbs += __builtin_fabs(e);
    }

    // a block's error sums, in a fixed order; true in the thread that has them
    __device__ __forceinline__ bool blockSums(double eRaw, double ePos, double eAbs, double (&red)[3][kSweepThreads / 64], double (&sum)[3])
    {
        eRaw = waveSum(eRaw);
        ePos = waveSum(ePos);
        eAbs = waveSum(eAbs);
        const uint32_t w = threadIdx.x >> 6;
        if ((threadIdx.x & 63u) == 0) { red[0][w] = eRaw; red[1][w] = ePos; red[2][w] = eAbs; }
        __syncthreads();
        if (threadIdx.x != 0) { return false; }
        for (int r = 0; r < 3; r++)
        {
            sum[r] = 0.0;
            for (uint32_t q = 0; q < kSweepThreads / 64; q++) { sum[r] += red[r][q]; }
        }
        return true;
    }

    // a neighbor of a Jacobi sweep: position and a^p
    struct SweepRec
    {
        float x, y, z, ax, ay, az;
    };

    // the FR terms of a Jacobi sweep
    __device__ __forceinline__ void relaxedFR(const Dev& d, const Lists& l, const Consts& k, const float4& at, float axi, float ayi, float azi,
        float& sb)
    {
        visit(l.list(d, REL_FR), [&](uint32_t j)
        {
            const float4 rj = d.rpos[j];
            const float dx = at.x - rj.x, dy = at.y - rj.y, dz = at.z - rj.z;
            const float f = kgFactor(dist2(dx, dy, dz), k);
            const float sv = __builtin_fmaf(axi, f * dx, __builtin_fmaf(ayi, f * dy, azi * (f * dz)));
            sb += rj.w * sv;
        });
    }

    // the relaxed pressure from the sums over fluid and boundary, and the predicted density error
    __device__ __forceinline__ float relaxedOf(const Consts& k, float sf, float sb, float p, float src, float diag, float& pred)
    {
        const float sys = k.dtsq * (sf + sb);
        const float resid = src - sys;
        pred = sys - src;
        const bool valid = __builtin_fabsf(diag) > 1e-7f;
        return vmax(0.0f, valid ? __builtin_fmaf(k.omega, resid / diag, p) : 0.0f);
    }

    // the relaxed pressure of a particle at `at` with acceleration ai and pressure p, and its predicted
    // density error; hp and ha hold the halo as (x, y, z, a^p x | a^p y, a^p z), 24 KB per block: six
    // blocks per CU; recOf(j) in a block without one
    template <bool kFast, typename RecOf>
    __device__ __forceinline__ float relaxedAt(const Dev& d, const Lists& l, const SlotList& slots, const Halo& h, const float4* hp,
        const float2* ha, const Consts& k, const float4& at, const float4& ai, float p, float src, float diag, RecOf&& recOf,
        float& pred)
    {
        const float xi = at.x, yi = at.y, zi = at.z, axi = ai.x, ayi = ai.y, azi = ai.z;
        float sf = 0.0f;
        const auto ffTerm = [&](float xj, float yj, float zj, float axj, float ayj, float azj, uint32_t q, auto shortFlag)
        {
            constexpr bool kShort = decltype(shortFlag)::value;
            const float dx = xi - xj, dy = yi - yj, dz = zi - zj;
            const float d2 = dist2(dx, dy, dz);
            const float kg = kShort ? addUlps(kgShort(d2, k), q) : kgFactor<kFast>(d2, k);
            const float sv = __builtin_fmaf(axi - axj, dx, __builtin_fmaf(ayi - ayj, dy, (azi - azj) * dz));
            sf = __builtin_fmaf(kg, sv, sf);
        };
        const auto haloLoad = [&](uint32_t q)
        {
            const float4 pj = recAt(hp, q);
            const float2 aj = recAt(ha, q);
            return SweepRec{ pj.x, pj.y, pj.z, pj.w, aj.x, aj.y };
        };
        const auto fromHalo = [&](uint32_t q, auto shortFlag)
        {
            const SweepRec r = haloLoad(q & kSlotMask);
            ffTerm(r.x, r.y, r.z, r.ax, r.ay, r.az, q, shortFlag);
        };
        if (kFast && h.ulps) { visitSlots(slots, [&](uint32_t q, uint32_t) { fromHalo(q, Flag<true>{}); }); }
        else if (h.any) { visitSlots(slots, [&](uint32_t q, uint32_t) { fromHalo(q, Flag<false>{}); }); }
        else
        {
            visit(l.list(d, REL_FF), [&](uint32_t j)
            {
                const SweepRec r = recOf(j);
                ffTerm(r.x, r.y, r.z, r.ax, r.ay, r.az, 0u, Flag<false>{});
            });
        }
        sf *= k.mass;
        float sb = 0.0f;
        visitGather(d, l, REL_FB, [&](uint32_t j) { return d.bpos[j]; }, [&](const float4& bj)
        {
            const float dx = xi - bj.x, dy = yi - bj.y, dz = zi - bj.z;
            const float f = kgFactor<kFast>(dist2(dx, dy, dz), k);
            const float sv = __builtin_fmaf(axi, f * dx, __builtin_fmaf(ayi, f * dy, azi * (f * dz)));
            sb += bj.w * sv;
        });
        relaxedFR(d, l, k, at, axi, ayi, azi, sb);
        return relaxedOf(k, sf, sb, p, src, diag, pred);
    }

    // one tile of a Jacobi sweep; nTot is the number of tiles (the stride of the error partials)
    template <bool kFast>
    __device__ __forceinline__ void jacobiTile(const Dev& d, uint32_t blk, uint32_t nTot)
    {
        __shared__ double red[3][kSweepThreads / 64];
        __shared__ float4 hp[kHaloMax];
        __shared__ float2 ha[kHaloMax];
        const Lists l = listsAt(d, blk);
        const SlotList slots = slotsOf(d, l);
        const Halo h = haloOf(d, blk);
        const uint32_t sc = uniformLoad(&d.blockScene[blk]);
        const Consts k = uniformLoad(&d.consts[sc]);
        const Scene S = uniformLoad(&d.scenes[sc]);
        // the scene's flags were written by an earlier launch: every thread reads the same values
        if (d.solve[sc].converged) { return; }
        const bool compute = d.solve[sc].compute != 0u;
        // (positions only: the pressures this launch writes into pos.w are not read here)
        const uint32_t i = l.i;
        const float4 pi = d.pos[i], ai = d.ap[i];
        const float src = d.source[i], diag = d.diag[i];
        stageHalo(h, [&](uint32_t j) { return Pair4{ d.pos[j], d.ap[j] }; }, [&](uint32_t q, const Pair4& r)
        {
            hp[q] = make_float4(r.a.x, r.a.y, r.a.z, r.b.x);
            ha[q] = make_float2(r.b.y, r.b.z);
        });
        __syncthreads();
        double eRaw = 0.0, ePos = 0.0, eAbs = 0.0;
        if (i - S.offF < S.nF)
        {
            float pred;
            d.pos[i].w = relaxedAt<kFast>(d, l, slots, h, hp, ha, k, pi, ai, pi.w, src, diag, [&](uint32_t j)
            {
                const float4 pj = d.pos[j], aj = d.ap[j];
                return SweepRec{ pj.x, pj.y, pj.z, aj.x, aj.y, aj.z };
            }, pred);
            const bool valid = __builtin_fabsf(diag) > 1e-7f;
            if (compute && valid) { addError(pred, k, eRaw, ePos, eAbs); }
        }
        if (blk == S.blk0 && threadIdx.x == 0) { d.solve[sc].pending = 1u; }
        if (!compute) { return; }
        double sum[3];
        if (blockSums(eRaw, ePos, eAbs, red, sum))
        {
            for (int r = 0; r < 3; r++) { d.errPartial[static_cast<size_t>(r) * nTot + blk] = sum[r]; }
        }
    }

    template <bool kFast>
    __global__ void __launch_bounds__(kSweepThreads) TSP_WAVES_ATTR(TSP_TUNE_JACOBI_WAVES) kJacobi(Dev d, uint32_t nTiles)
    {
        if (stopped(d)) { return; }
        jacobiTile<kFast>(d, xcdBlock(), nTiles);
    }

    // --- the whole solve in one launch, for a context of few blocks ---
    // A sweep of 64,000 particles is two launches of 9 to 10 us with 4 us between them, of which the pair
    // sums take a third: the rest is launch, drain and the loads that every launch repeats. Here the blocks
    // stay: positions, list heads and the particle's own values are loaded once, each half sweep
    // gathers only what the other half wrote, and the blocks of a scene meet at a barrier after it (the
    // scenes are independent). The bookkeeping of a sweep is done by every block for itself from the
    // partial sums, in the order of finalizeSweep, beside the next accelerations; those of the sweep that
    // converged are the final ones. No host read, and the same bits. A sweep of 64,000 particles: 27 us launch
    // by launch, 11.8 here (a fifth each the two sums, a quarter each the two barriers); 4,096 particles: 17
    // and 10.5. With two blocks per CU (111,000 particles) it was no faster than the launches.
    // The blocks must all be resident: the host asks for at most one per CU, and the first barrier, before
    // anything is written, gives up when other work keeps some block out for kEntrySpins polls: the scene's
    // blocks then leave together, and the host runs the sweeps launch by launch. Past the first
    // barrier every block of the scene is running.
    constexpr uint32_t kEntrySpins = 4000;
    constexpr uint32_t kBarSpins = 1u << 20;
    // offsets into a scene's entry words: arrivals, and the outcome
    constexpr uint32_t kBarArrived = 0, kBarEntry = kBarLine;
    constexpr uint32_t kEntryOpen = 0, kEntryGo = 1, kEntryGaveUp = 2;

    // What another block reads in the same launch goes past the L2 of the block's XCD both ways: device-scope
    // words.
    __device__ __forceinline__ void putWord(float* p, float v)
    {
        __hip_atomic_store(reinterpret_cast<uint32_t*>(p), __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ float getWord(const float* p)
    {
        return __uint_as_float(__hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
    __device__ __forceinline__ void putAcc(float4* p, float x, float y, float z)
    {
        unsigned long long* w = reinterpret_cast<unsigned long long*>(p);
        __hip_atomic_store(w, static_cast<unsigned long long>(__float_as_uint(y)) << 32 | __float_as_uint(x), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(w + 1, static_cast<unsigned long long>(__float_as_uint(z)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ float4 getAcc(const float4* p)
    {
        const unsigned long long* w = reinterpret_cast<const unsigned long long*>(p);
        const unsigned long long a = __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long b = __hip_atomic_load(w + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return make_float4(__uint_as_float(static_cast<uint32_t>(a)), __uint_as_float(static_cast<uint32_t>(a >> 32)),
                           __uint_as_float(static_cast<uint32_t>(b)), 0.0f);
    }

    // a value that is the same in every lane
    __device__ __forceinline__ float uniform(float v)
    {
        return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
    }

    // The n-th barrier (from 1) of a scene's blocks, in two halves. Arrival, all threads: every store before it
    // has reached memory (the wait is for the stores themselves: they carry the device scope, no cache
    // holds them back) before the block raises its flag to n. A flag per block, all read by the waiting
    // wave at once, in as many copies as there are XCDs (readers of one line queue up): from the last of 250
    // arrivals on 3,700 cycles at least; 5,000 with one copy, 6,300 with a counter and a word that says go.
    // An agent-scope release here (and an acquire after the wait) would write back and invalidate the L2s, which
    // hold nothing of what is exchanged: 64,000 particles, 100 sweeps: 1,466 us a step, 2,776 (3,060) with them.
    __device__ __forceinline__ void arriveScene(uint32_t* flags, uint32_t blk, uint32_t n)
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        const uint32_t copy = threadIdx.x - (kSweepThreads - 64u);
        if (copy < kFlagCopies)
        {
            __hip_atomic_store(&flags[copy * kSolveBlocksMost + blk], n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }

    // The wait for the others, all threads (the last wave polls). False when the block gave up waiting
    // (never expected).
    __device__ __forceinline__ bool meetScene(const uint32_t* flags, const Scene& S, uint32_t n, uint32_t* fail)
    {
        __shared__ uint32_t met;
        if (threadIdx.x >= kSweepThreads - 64u)
        {
            constexpr uint32_t kPolls = kSolveBlocksMost / 64u;
            const uint32_t lane = threadIdx.x & 63u;
            flags += (blockIdx.x & (kFlagCopies - 1u)) * kSolveBlocksMost + S.blk0;
            uint32_t spins = 0;
            for (;;)
            {
                uint32_t f[kPolls];
                for (uint32_t q = 0; q < kPolls; q++)
                {
                    const uint32_t b = q * 64u + lane;
                    f[q] = b < S.nBlk ? __hip_atomic_load(&flags[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : n;
                }
                bool here = true;
                for (uint32_t q = 0; q < kPolls; q++) { here = here && f[q] >= n; }
                if (__ballot(!here) == 0ull) { break; }
                if (++spins > kBarSpins) { break; }
            }
            if (lane == 0u)
            {
                met = spins <= kBarSpins;
                if (spins > kBarSpins) { atomicOr(fail, 1u); }
            }
        }
        __syncthreads();
        return met != 0u;
    }

    // the first barrier: true for all blocks of the scene, or false for all
    __device__ __forceinline__ bool enterScene(uint32_t* bar, uint32_t nBlk)
    {
        __shared__ uint32_t outcome;
        if (threadIdx.x == 0)
        {
            uint32_t seen = kEntryOpen;
            const uint32_t before = __hip_atomic_fetch_add(&bar[kBarArrived], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (before + 1u == nBlk)
            {
                // (seen comes back as what was there: gave up, or open)
                if (__hip_atomic_compare_exchange_strong(&bar[kBarEntry], &seen, kEntryGo, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT)) { seen = kEntryGo; }
            }
            else
            {
                for (uint32_t spins = 0; seen == kEntryOpen; spins++)
                {
                    seen = __hip_atomic_load(&bar[kBarEntry], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (seen == kEntryOpen && spins >= kEntrySpins)
                    {
                        if (__hip_atomic_compare_exchange_strong(&bar[kBarEntry], &seen, kEntryGaveUp, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                                 __HIP_MEMORY_SCOPE_AGENT)) { seen = kEntryGaveUp; }
                    }
                }
            }
            outcome = seen;
        }
        __syncthreads();
        return outcome == kEntryGo;
    }

    // What a thread keeps of its pairs for the whole solve, in a wave whose FF lists have at most kKeepFF
    // entries: the FF entries' distances, gradient factors and halo slots in registers, and the FB entries'
    // gradients and psi in LDS (the first kRowsFB entries; further ones in d.fbGrad, each read by the
    // thread that wrote it). A half sweep then gathers 4 or 12 bytes per pair from LDS instead of 16 or 24, which is what the sums
    // are bound by (64 records of 16 bytes at random places take the LDS about 25 cycles, three times what
    // they take in a row), and computes a third.
    constexpr uint32_t kKeepFF = 40;
    constexpr uint32_t kRowsFB = 20;

    struct Kept
    {
        float dx[kKeepFF], dy[kKeepFF], dz[kKeepFF], kg[kKeepFF];
        uint32_t slots[kKeepFF / 2];   // two entries each
        uint32_t n, pitch, nAll;       // of the FF list, of its slice, and of the wave's shortest list
        uint32_t nB;
        float4* fb;                    // the lane's FB record in row 0, in LDS; from row kRowsFB on in memory
        float4* fbMore;

        __device__ __forceinline__ uint32_t slot(uint32_t q) const { return (q & 1u) ? slots[q / 2u] >> 16 : slots[q / 2u] & 0xffffu; }

        template <bool kFast>
        __device__ __forceinline__ void fill(const Dev& d, const Lists& l, const SlotList& s, const Halo& h, const float4* hp,
            float4* rows, const Consts& k, const float4& at)
        {
            n = s.n;
            pitch = s.pitch;
            uint32_t m = n;
            for (int o = 32; o > 0; o >>= 1) { m = min(m, static_cast<uint32_t>(__shfl_xor(static_cast<int>(m), o, 64))); }
            nAll = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(m)));
            const auto put = [&](uint32_t q, uint32_t entry, auto shortFlag)
            {
                constexpr bool kShort = decltype(shortFlag)::value;
                const float4& pj = recAt(hp, entry & kSlotMask);
                dx[q] = at.x - pj.x; dy[q] = at.y - pj.y; dz[q] = at.z - pj.z;
                const float d2 = dist2(dx[q], dy[q], dz[q]);
                kg[q] = kShort ? addUlps(kgShort(d2, k), entry) : kgFactor<kFast>(d2, k);
            };
#pragma unroll
            for (uint32_t q = 0; q < kKeepFF; q += 2u)
            {
                // (an entry past the list repeats the first one, or slot 0, and is not used)
                uint32_t e0 = s.p[(q < n ? q : 0u) * kSlice], e1 = s.p[(q + 1u < n ? q + 1u : 0u) * kSlice];
                e0 = n ? e0 : 0u;
                e1 = n ? e1 : 0u;
                if (kFast && h.ulps) { put(q, e0, Flag<true>{}); put(q + 1u, e1, Flag<true>{}); }
                else { put(q, e0, Flag<false>{}); put(q + 1u, e1, Flag<false>{}); }
                slots[q / 2u] = (e0 & kSlotMask) | (e1 & kSlotMask) << 16;
            }
            nB = l.n[REL_FB];
            fb = rows;
            fbMore = d.fbGrad + l.m[REL_FB].offset + l.lane;
            uint32_t row = 0;
            visitGather(d, l, REL_FB, [&](uint32_t j) { return d.bpos[j]; }, [&](const float4& bj)
            {
                const float dx = at.x - bj.x, dy = at.y - bj.y, dz = at.z - bj.z;
                const float f = kgFactor<kFast>(dist2(dx, dy, dz), k);
                const float4 g = make_float4(f * dx, f * dy, f * dz, bj.w);
                if (row < kRowsFB) { fb[row * kBlock] = g; } else { fbMore[row * kSlice] = g; }
                row++;
            });
        }

        // visits the FF entries in list order, as use(q, load(slot)); four entries load while the four before
        // are summed
        template <typename Load, typename Use>
        __device__ __forceinline__ void visitFF(Load&& load, Use&& use)
        {
            using R = decltype(load(0u));
            // (opaque here: unpacked ahead of the sweeps' loop they would take twice the registers)
#pragma unroll
            for (uint32_t q = 0; q < kKeepFF / 2u; q++) { asm volatile("" : "+v"(slots[q])); }
            asm volatile("" : "+v"(n));
            R r0 = load(slot(0u)), r1 = load(slot(1u)), r2 = load(slot(2u)), r3 = load(slot(3u));
#pragma unroll
            for (uint32_t q = 0; q < kKeepFF; q += 4u)
            {
                if (q < pitch)
                {
                    R n0{}, n1{}, n2{}, n3{};
                    if (q + 4u < kKeepFF)
                    {
                        n0 = load(slot(q + 4u)); n1 = load(slot(q + 5u)); n2 = load(slot(q + 6u)); n3 = load(slot(q + 7u));
                    }
                    if (q + 4u <= nAll) { use(q, r0); use(q + 1u, r1); use(q + 2u, r2); use(q + 3u, r3); }
                    else
                    {
                        if (q < n) { use(q, r0); }
                        if (q + 1u < n) { use(q + 1u, r1); }
                        if (q + 2u < n) { use(q + 2u, r2); }
                        if (q + 3u < n) { use(q + 3u, r3); }
                    }
                    r0 = n0; r1 = n1; r2 = n2; r3 = n3;
                }
            }
        }

        template <typename Use>
        __device__ __forceinline__ void visitFB(Use&& use) const
        {
            uint32_t q = 0;
            const uint32_t near = min(nB, kRowsFB);
            for (; q + 4u <= near; q += 4u)
            {
                const float4 b0 = fb[q * kBlock], b1 = fb[(q + 1u) * kBlock], b2 = fb[(q + 2u) * kBlock], b3 = fb[(q + 3u) * kBlock];
                use(b0); use(b1); use(b2); use(b3);
            }
            for (; q < near; q++) { use(fb[q * kBlock]); }
            for (; q < nB; q++) { use(fbMore[q * kSlice]); }
        }

        // pressureAt and relaxedAt from what is kept
        __device__ __forceinline__ void pressure(const Dev& d, const Lists& l, const float* hw, const Consts& k, const float4& p4,
            float (&a)[3])
        {
            const float pi = p4.w;
            float sx = 0.0f, sy = 0.0f, sz = 0.0f;
            visitFF([&](uint32_t e) { return hw[e >> kSlotShift]; }, [&](uint32_t q, float pj)
            {
                const float coeff = (pi + pj) * kg[q];
                sx = __builtin_fmaf(coeff, dx[q], sx);
                sy = __builtin_fmaf(coeff, dy[q], sy);
                sz = __builtin_fmaf(coeff, dz[q], sz);
            });
            float ax = sx * k.presOuterFF, ay = sy * k.presOuterFF, az = sz * k.presOuterFF;
            visitFB([&](const float4& g)
            {
                const float coeff = k.presOuterB * g.w * pi;
                ax = __builtin_fmaf(coeff, g.x, ax);
                ay = __builtin_fmaf(coeff, g.y, ay);
                az = __builtin_fmaf(coeff, g.z, az);
            });
            pressureFR(d, l, k, p4, ax, ay, az);
            a[0] = 0.0f - ax; a[1] = 0.0f - ay; a[2] = 0.0f - az;
        }

        __device__ __forceinline__ float relaxed(const Dev& d, const Lists& l, const float* hw, const float2* ha, const Consts& k,
            const float4& p4, const float (&a)[3], float src, float diag, float& pred)
        {
            struct Acc
            {
                float x;
                float2 yz;
            };
            float sf = 0.0f;
            visitFF([&](uint32_t e) { return Acc{ hw[e >> kSlotShift], recAt(ha, e) }; }, [&](uint32_t q, const Acc& r)
            {
                sf = __builtin_fmaf(kg[q], __builtin_fmaf(a[0] - r.x, dx[q],
                                    __builtin_fmaf(a[1] - r.yz.x, dy[q], (a[2] - r.yz.y) * dz[q])), sf);
            });
            sf *= k.mass;
            float sb = 0.0f;
            visitFB([&](const float4& g)
            {
                sb += g.w * __builtin_fmaf(a[0], g.x, __builtin_fmaf(a[1], g.y, a[2] * g.z));
            });
            relaxedFR(d, l, k, p4, a[0], a[1], a[2], sb);
            return relaxedOf(k, sf, sb, p4.w, src, diag, pred);
        }
    };

    // held: a scene whose entry waits for one block more than it has, and so gives up (none: kEmpty32)
    template <bool kFast>
    __global__ void __launch_bounds__(kSweepThreads) __attribute__((amdgpu_waves_per_eu(1, 1))) kSolve(Dev d, uint32_t held)
    {
        __shared__ double red[3][kSweepThreads / 64];
        __shared__ double part[3][kSolveBlocksMost];
        __shared__ double sums[3];
        __shared__ float4 hp[kHaloMax];
        __shared__ float2 ha[kHaloMax];
        __shared__ float hw[kHaloMax];   // hp's last word by itself
        __shared__ float4 fbRows[kRowsFB * kBlock];
        const uint32_t nTot = gridDim.x, t = threadIdx.x;
        const uint32_t blk = xcdBlock();
        const Lists l = listsAt(d, blk);
        const SlotList slots = slotsOf(d, l);
        Halo h = haloOf(d, blk);
        const uint32_t sc = uniformLoad(&d.blockScene[blk]);
        const Consts k = uniformLoad(&d.consts[sc]);
        const Scene S = uniformLoad(&d.scenes[sc]);
        const uint32_t i = l.i;
        float4 p4 = d.pos[i];
        const float src = d.source[i], diag = d.diag[i];
        const bool active = i - S.offF < S.nF;
        stageHalo(h, [&](uint32_t j) { return d.pos[j]; }, [&](uint32_t q, const float4& r) { hp[q] = r; hw[q] = r.w; });
        // the state that solverInit left (the rest of it is 0); every thread keeps it
        Solve s{};
        s.iters = d.solve[sc].iters;
        s.compute = d.solve[sc].compute;
        uint32_t* bar = d.solveBar + static_cast<size_t>(sc) * kBarWords;
        if (!enterScene(bar, S.nBlk + (sc == held ? 1u : 0u))) { return; }   // (a barrier: the halo is staged)
        Kept kept;
        const bool keep = h.any && __ballot(active && l.n[REL_FF] > kKeepFF) == 0ull;
        if (keep && active) { kept.fill<kFast>(d, l, slots, h, hp, fbRows + t, k, p4); }
        const bool valid = __builtin_fabsf(diag) > 1e-7f;
        uint32_t meet = 0;
        for (;;)
        {
            const bool pending = meet != 0u;
            // (opaque: the addresses are made in each round)
            for (uint32_t u = 0; u < Halo::kPer; u++) { asm volatile("" : "+v"(h.j[u])); }
            if (pending)
            {
                // the pressures of the sweep before and, if it took its errors, all blocks' sums of them
                float w[Halo::kPer];
                for (uint32_t u = 0; u < Halo::kPer; u++)
                {
                    if (u * kBlock < h.count) { w[u] = getWord(&d.pos[u * kBlock + t < h.count ? h.j[u] : 0u].w); }
                }
                if (s.compute)
                {
                    for (int r = 0; r < 3; r++)
                    {
                        const unsigned long long* from = reinterpret_cast<const unsigned long long*>(d.errPartial)
                                                       + static_cast<size_t>(r) * nTot + S.blk0;
                        for (uint32_t b = t; b < kSolveBlocksMost; b += kSweepThreads)
                        {
                            if (b < S.nBlk)
                            {
                                part[r][b] = __longlong_as_double(static_cast<long long>(
                                    __hip_atomic_load(&from[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)));
                            }
                        }
                    }
                }
                for (uint32_t u = 0; u < Halo::kPer; u++) { if (u * kBlock + t < h.count) { hp[u * kBlock + t].w = w[u]; hw[u * kBlock + t] = w[u]; } }
                __syncthreads();
            }
            float a[3] = { 0.0f, 0.0f, 0.0f };
            if (active)
            {
                if (keep) { kept.pressure(d, l, hw, k, p4, a); }
                else
                {
                    pressureAt<kFast>(d, l, slots, h, hp, k, p4, [&](uint32_t j)
                    {
                        const float4 q = d.pos[j];
                        return make_float4(q.x, q.y, q.z, getWord(&d.pos[j].w));
                    }, a);
                }
                putAcc(&d.ap[i], a[0], a[1], a[2]);
            }
            arriveScene(d.solveFlag, blk, ++meet);
            if (pending)
            {
                // finalizeSweep's sums, in its order (a wave per sum), and its decision
                s.sweeps++;
                if (s.compute)
                {
                    const uint32_t r = t >> 6;
                    if (r < 3u)
                    {
                        double v[kSweepThreads / 64];
                        for (uint32_t w = 0; w < kSweepThreads / 64; w++)
                        {
                            v[w] = 0.0;
                            for (uint32_t b = w * 64u + (t & 63u); b < S.nBlk; b += kSweepThreads) { v[w] += part[r][b]; }
                        }
                        for (uint32_t w = 0; w < kSweepThreads / 64; w++) { v[w] = waveSum(v[w]); }
                        double sum = v[0];
                        for (uint32_t w = 1; w < kSweepThreads / 64; w++) { sum += v[w]; }
                        if ((t & 63u) == 0u) { sums[r] = sum; }
                    }
                    __syncthreads();
                    const float n = static_cast<float>(S.nF);
                    s.avgRaw = uniform(static_cast<float>(sums[0]) / n);
                    s.avgPos = uniform(static_cast<float>(sums[1]) / n);
                    s.avgAbs = uniform(static_cast<float>(sums[2]) / n);
                    if (blk == S.blk0 && t == 0)
                    {
                        Solve& out = d.solve[sc];
                        out.sumRaw = sums[0]; out.sumPos = sums[1]; out.sumAbs = sums[2];
                        out.avgRaw = s.avgRaw; out.avgPos = s.avgPos; out.avgAbs = s.avgAbs;
                    }
                }
                if (terminated(s, k)) { break; }
                s.iters++;
                s.compute = (s.iters >= k.minIters && (k.termCond != 0 || terminated(s, k))) ? 1u : 0u;
            }
            if (!meetScene(d.solveFlag, S, meet, &d.status->scanFail)) { return; }
            {
                float4 w[Halo::kPer];
                for (uint32_t u = 0; u < Halo::kPer; u++)
                {
                    if (u * kBlock < h.count) { w[u] = getAcc(&d.ap[u * kBlock + t < h.count ? h.j[u] : 0u]); }
                }
                for (uint32_t u = 0; u < Halo::kPer; u++)
                {
                    if (u * kBlock + t < h.count)
                    {
                        hp[u * kBlock + t].w = w[u].x;
                        hw[u * kBlock + t] = w[u].x;
                        ha[u * kBlock + t] = make_float2(w[u].y, w[u].z);
                    }
                }
                __syncthreads();
            }
            double eRaw = 0.0, ePos = 0.0, eAbs = 0.0;
            if (active)
            {
                float pred;
                if (keep) { p4.w = kept.relaxed(d, l, hw, ha, k, p4, a, src, diag, pred); }
                else
                {
                    p4.w = relaxedAt<kFast>(d, l, slots, h, hp, ha, k, p4, make_float4(a[0], a[1], a[2], 0.0f), p4.w, src, diag, [&](uint32_t j)
                    {
                        const float4 pj = d.pos[j], aj = getAcc(&d.ap[j]);
                        return SweepRec{ pj.x, pj.y, pj.z, aj.x, aj.y, aj.z };
                    }, pred);
                }
                putWord(&d.pos[i].w, p4.w);
                if (s.compute && valid) { addError(pred, k, eRaw, ePos, eAbs); }
            }
            if (s.compute)
            {
                double sum[3];
                if (blockSums(eRaw, ePos, eAbs, red, sum))
                {
                    for (int r = 0; r < 3; r++)
                    {
                        __hip_atomic_store(reinterpret_cast<unsigned long long*>(d.errPartial) + static_cast<size_t>(r) * nTot + blk,
                                           static_cast<unsigned long long>(__double_as_longlong(sum[r])), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            }
            arriveScene(d.solveFlag, blk, ++meet);
            if (!meetScene(d.solveFlag, S, meet, &d.status->scanFail)) { return; }
        }
        if (blk == S.blk0 && t == 0)
        {
            Solve& out = d.solve[sc];
            out.iters = s.iters; out.sweeps = s.sweeps; out.compute = s.compute; out.converged = 1u;
        }
    }

    // the bookkeeping of the last sweep of a group, one block per scene, before the host reads
    // the solver states; nTot is the grid size of the sweeps
    __global__ void __launch_bounds__(kSweepThreads) kFinalize(Dev d, uint32_t nTot)
    {
        if (stopped(d)) { return; }
        finalizeSweep(d, blockIdx.x, nTot);
    }

    __global__ void __launch_bounds__(kBlock) kIntegration(Dev d)
    {
        if (stopped(d)) { return; }
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        const uint32_t sc = d.blockScene[blockIdx.x];
        const Consts& k = d.consts[sc];
        if (i - d.scenes[sc].offF >= d.scenes[sc].nF) { return; }
        const float4 a = d.ap[i], v = d.vp[i], p = d.pos[i];
        const float vx = __builtin_fmaf(k.dt, a.x, v.x);
        const float vy = __builtin_fmaf(k.dt, a.y, v.y);
        const float vz = __builtin_fmaf(k.dt, a.z, v.z);
        d.vel[i] = make_float4(vx, vy, vz, d.vel[i].w);
        d.pos[i] = make_float4(__builtin_fmaf(k.dt, vx, p.x), __builtin_fmaf(k.dt, vy, p.y), __builtin_fmaf(k.dt, vz, p.z), p.w);
    }

    // ----------------------------------------------------------------------------------------
    // rigid bodies; the body state is field-major: rb[field * nRB + body] (rbv)

    // UpdateRigidParticles(predicted), cpu_backend.cpp:2009-2063
    __global__ void __launch_bounds__(kBlock) kRigidUpdate(Dev d, bool predicted)
    {
        if (stopped(d)) { return; }
        const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
        if (i < d.nR) { rigidUpdateOne(d, i, predicted); }
    }

    // AccumulateRigidParticleNonPressureForces_ChunkedSELL / ...PressureForces (sph_solver.cpp:1151-1223,
    // :1717-1778): reaction of the fluid neighbors of each rigid particle
    __global__ void __launch_bounds__(kBlock) kRigidForces(Dev d, bool pressure)
    {
        if (stopped(d)) { return; }
        // one wave per rigid particle: the lanes compute 64 pairs' coefficients and gradients at
        // once, then every lane folds them in list order (the single-thread sum, term by term)
        const uint32_t i = (blockIdx.x * kBlock + threadIdx.x) >> 6;
        const uint32_t lane = threadIdx.x & 63u;
        if (i >= d.nR) { return; }
        const Consts& k = d.consts[d.bodyScene[d.rbody[i]]];
        const float4 ri = d.rpos[i], ui = d.rvel[i];
        const float xi = ri.x, yi = ri.y, zi = ri.z;
        float fx = 0.0f, fy = 0.0f, fz = 0.0f;
        const uint32_t q0 = d.rfOff[i], q1 = d.rfOff[i + 1];
        for (uint32_t base = q0; base < q1; base += 64)
        {
            const uint32_t q = base + lane;
            float fc = 0.0f, gx = 0.0f, gy = 0.0f, gz = 0.0f;
            if (q < q1)
            {
                const uint32_t j = d.rfIdx[q];
                const float4 pj = d.pos[j];
                const float dx = pj.x - xi, dy = pj.y - yi, dz = pj.z - zi;
                kgScalar(dx, dy, dz, k, gx, gy, gz);
                if (pressure)
                {
                    fc = k.mass * k.presOuterB * ri.w * pj.w;
                }
                else
                {
                    const float4 vj = d.vel[j];
                    const float dvx = vj.x - ui.x, dvy = vj.y - ui.y, dvz = vj.z - ui.z;
                    const float dot = __builtin_fmaf(dvx, dx, __builtin_fmaf(dvy, dy, dvz * dz));
                    const float d2 = dist2(dx, dy, dz);
                    const float coeff = (ui.w * dot) / (d2 + k.hsqEps);
                    fc = -k.mass * k.visB * coeff;
                }
            }
            const uint32_t n = min(64u, q1 - base);
            for (uint32_t l = 0; l < n; l++)
            {
                const float c = __shfl(fc, static_cast<int>(l), 64);
                fx = __builtin_fmaf(c, __shfl(gx, static_cast<int>(l), 64), fx);
                fy = __builtin_fmaf(c, __shfl(gy, static_cast<int>(l), 64), fy);
                fz = __builtin_fmaf(c, __shfl(gz, static_cast<int>(l), 64), fz);
            }
        }
        if (lane != 0) { return; }
        if (pressure) { d.rfx[i] += fx; d.rfy[i] += fy; d.rfz[i] += fz; }
        else { d.rfx[i] = fx; d.rfy[i] = fy; d.rfz[i] = fz; }
    }

    __device__ __forceinline__ bool normalize3(float& x, float& y, float& z)
    {
        const float len = __builtin_sqrtf(__builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z)));
        if (len <= 1e-12f || !__builtin_isfinite(len)) { return false; }
        const float inv = 1.0f / len;
        x *= inv; y *= inv; z *= inv;
        return true;
    }

    __device__ __forceinline__ float dot3(float ax, float ay, float az, float bx, float by, float bz)
    {
        return __builtin_fmaf(ax, bx, __builtin_fmaf(ay, by, az * bz));
    }

    // IntegrateRigidBodies, cpu_backend.cpp:2237-2303, one body
    __device__ __forceinline__ void rigidIntegrateOne(const Dev& d, uint32_t b)
    {
        const Consts& k = d.consts[d.bodyScene[b]];
        const uint32_t nb = d.nRB;
        float* rb = d.rb;
        for (int a = 0; a < 3; a++)
        {
            rb[(RB_VX + a) * nb + b] = d.rbPred[a * nb + b];
            rb[(RB_LX + a) * nb + b] = d.rbPred[(3 + a) * nb + b];
        }
        for (int a = 0; a < 3; a++) { rb[(RB_XCM + a) * nb + b] += k.dt * rb[(RB_VX + a) * nb + b]; }
        const float wx = d.rbPred[6 * nb + b], wy = d.rbPred[7 * nb + b], wz = d.rbPred[8 * nb + b];
        rb[(RB_WX + 0) * nb + b] = wx;
        rb[(RB_WX + 1) * nb + b] = wy;
        rb[(RB_WX + 2) * nb + b] = wz;
        float A[9];
        for (int q = 0; q < 9; q++) { A[q] = rb[(RB_A00 + q) * nb + b]; }
        const float dt = k.dt;
        float N[9];
        N[0] = A[0] + dt * (-wz * A[3] + wy * A[6]);
        N[1] = A[1] + dt * (-wz * A[4] + wy * A[7]);
        N[2] = A[2] + dt * (-wz * A[5] + wy * A[8]);
        N[3] = A[3] + dt * (wz * A[0] - wx * A[6]);
        N[4] = A[4] + dt * (wz * A[1] - wx * A[7]);
        N[5] = A[5] + dt * (wz * A[2] - wx * A[8]);
        N[6] = A[6] + dt * (-wy * A[0] + wx * A[3]);
        N[7] = A[7] + dt * (-wy * A[1] + wx * A[4]);
        N[8] = A[8] + dt * (-wy * A[2] + wx * A[5]);
        float b1x = N[0], b1y = N[3], b1z = N[6];
        float b2x = N[1], b2y = N[4], b2z = N[7];
        float b3x = N[2], b3y = N[5], b3z = N[8];
        bool ok = normalize3(b1x, b1y, b1z);
        const float d12 = dot3(b1x, b1y, b1z, b2x, b2y, b2z);
        b2x -= d12 * b1x; b2y -= d12 * b1y; b2z -= d12 * b1z;
        ok = ok && normalize3(b2x, b2y, b2z);
        const float d13 = dot3(b1x, b1y, b1z, b3x, b3y, b3z);
        const float d23 = dot3(b2x, b2y, b2z, b3x, b3y, b3z);
        b3x -= d13 * b1x + d23 * b2x;
        b3y -= d13 * b1y + d23 * b2y;
        b3z -= d13 * b1z + d23 * b2z;
        ok = ok && normalize3(b3x, b3y, b3z);
        if (!ok) { atomicOr(&d.solve[d.bodyScene[b]].rigidDegenerate, 1u); return; }
        const float out[9] = { b1x, b2x, b3x, b1y, b2y, b3y, b1z, b2z, b3z };
        for (int q = 0; q < 9; q++) { rb[(RB_A00 + q) * nb + b] = out[q]; }
    }

    // ClearRigidForcesAndAddGravity and ReduceRigidParticleForcesToBody (cpu_backend.cpp:2065-2172) of one
    // body, with FP64 sums, by its block of kBodyThreads; thread 0 writes the sums
    constexpr uint32_t kBodyThreads = 1024;

    __device__ __forceinline__ void rigidForceSums(const Dev& d, uint32_t b)
    {
        __shared__ double red[6][kBodyThreads];
        const uint32_t t = threadIdx.x;
        const uint32_t nb = d.nRB;
        const float a[9] = { rbv(d, RB_A00 + 0, b), rbv(d, RB_A00 + 1, b), rbv(d, RB_A00 + 2, b),
                             rbv(d, RB_A00 + 3, b), rbv(d, RB_A00 + 4, b), rbv(d, RB_A00 + 5, b),
                             rbv(d, RB_A00 + 6, b), rbv(d, RB_A00 + 7, b), rbv(d, RB_A00 + 8, b) };
        double acc[6] = { 0, 0, 0, 0, 0, 0 };
        for (uint32_t q = d.byBodyOff[b] + t; q < d.byBodyOff[b + 1]; q += kBodyThreads)
        {
            const uint32_t i = d.byBodyIdx[q];
            const float lx = d.rxrel[i], ly = d.ryrel[i], lz = d.rzrel[i];
            const float rx = __builtin_fmaf(a[0], lx, __builtin_fmaf(a[1], ly, a[2] * lz));
            const float ry = __builtin_fmaf(a[3], lx, __builtin_fmaf(a[4], ly, a[5] * lz));
            const float rz = __builtin_fmaf(a[6], lx, __builtin_fmaf(a[7], ly, a[8] * lz));
            const double fx = d.rfx[i], fy = d.rfy[i], fz = d.rfz[i];
            acc[0] += fx; acc[1] += fy; acc[2] += fz;
            acc[3] += static_cast<double>(ry) * fz - static_cast<double>(rz) * fy;
            acc[4] += static_cast<double>(rz) * fx - static_cast<double>(rx) * fz;
            acc[5] += static_cast<double>(rx) * fy - static_cast<double>(ry) * fx;
        }
        for (int f = 0; f < 6; f++) { red[f][t] = acc[f]; }
        __syncthreads();
        for (uint32_t o = kBodyThreads / 2; o >= 64u; o >>= 1)
        {
            if (t < o) { for (int f = 0; f < 6; f++) { red[f][t] += red[f][t + o]; } }
            __syncthreads();
        }
        if (t >= 64u) { return; }
        for (int f = 0; f < 6; f++)
        {
            // the last six halvings in the first wave (lanes past each half hold what is not used)
            double v = red[f][t];
            for (int o = 32; o > 0; o >>= 1) { v += __shfl_down(v, o, 64); }
            acc[f] = v;
        }
        if (t != 0u) { return; }
        const Consts& k = d.consts[d.bodyScene[b]];
        const float m = rbv(d, RB_MASS, b), mi = rbv(d, RB_MASS_INV, b);
        float g[6] = { 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f };
        if (!(m <= 0.0f || mi <= 0.0f)) { g[0] += m * k.gx; g[1] += m * k.gy; g[2] += m * k.gz; }
        for (int f = 0; f < 6; f++) { d.rbForce[f * nb + b] = g[f] + static_cast<float>(acc[f]); }
    }

    // A body's part of a step in one block: the force sums, the prediction, the integration and the body's
    // particles, whichever `parts` asks for, in this order. Each was a launch of 4 to 10 us of which little
    // more than the launch was needed. Where a body has more than kBodyParticles, the particles are updated by a
    // launch of their own: a block takes about 2 us per thousand of its body's. A step with one body of 2,044 /
    // 2,368 / 3,088 / 3,904 / 6,364 particles: 557 / 605 / 687 / 799 / 1,256 us together, 559 / 605 / 686 / 796 /
    // 1,246 apart; several bodies share the time of the largest: ten of 1,468 take 371 us together, 390 apart.
    constexpr uint32_t kBodyParticles = 2048;
    enum BodyParts { kBodySums = 1, kBodyPredict = 2, kBodyIntegrate = 4, kBodyUpdate = 8, kBodyUpdatePredicted = 16 };

    __global__ void __launch_bounds__(kBodyThreads) kRigidBody(Dev d, uint32_t parts)
    {
        if (stopped(d)) { return; }
        const uint32_t b = blockIdx.x;
        if (parts & kBodySums) { rigidForceSums(d, b); }
        if (threadIdx.x == 0u)
        {
            if (parts & kBodyPredict) { rigidPredictOne(d, b); }
            if (parts & kBodyIntegrate) { rigidIntegrateOne(d, b); }
        }
        if ((parts & (kBodyUpdate | kBodyUpdatePredicted)) == 0u) { return; }
        __syncthreads();   // (the body's new state, written by thread 0, is read by the block)
        for (uint32_t q = d.byBodyOff[b] + threadIdx.x; q < d.byBodyOff[b + 1]; q += kBodyThreads)
        {
            rigidUpdateOne(d, d.byBodyIdx[q], (parts & kBodyUpdatePredicted) != 0u);
        }
    }

    // ----------------------------------------------------------------------------------------
    // host launchers

    static inline uint32_t blocksOf(uint64_t n) { return static_cast<uint32_t>((n + kBlock - 1) / kBlock); }

    void launchDensity(hipStream_t s, const Dev& d)
    {
        if (!d.nF) { return; }
        if (d.fastPairs) { kDensity<true><<<blocksOf(d.nF), kBlock, 0, s>>>(d); }
        else { kDensity<false><<<blocksOf(d.nF), kBlock, 0, s>>>(d); }
    }
    void launchNonPressure(hipStream_t s, const Dev& d)
    {
        if (!d.nF) { return; }
        if (d.fastPairs) { kNonPressure<true><<<blocksOf(d.nF), kBlock, 0, s>>>(d); }
        else { kNonPressure<false><<<blocksOf(d.nF), kBlock, 0, s>>>(d); }
    }
    void launchSourceDiag(hipStream_t s, const Dev& d)
    {
        if (!d.nScenes) { return; }
        if (d.fastPairs) { kSourceDiag<true><<<blocksOf(d.nF) + 1u, kBlock, 0, s>>>(d); }
        else { kSourceDiag<false><<<blocksOf(d.nF) + 1u, kBlock, 0, s>>>(d); }
    }
    void launchPressureAcc(hipStream_t s, const Dev& d, bool sweep)
    {
        if (!d.nF) { return; }
        const uint32_t n = blocksOf(d.nF);
        if (d.fastPairs) { kPressureAcc<true><<<n, kSweepThreads, 0, s>>>(d, sweep, n); }
        else { kPressureAcc<false><<<n, kSweepThreads, 0, s>>>(d, sweep, n); }
    }
    void launchJacobi(hipStream_t s, const Dev& d)
    {
        if (!d.nF) { return; }
        const uint32_t n = blocksOf(d.nF);
        if (d.fastPairs) { kJacobi<true><<<n, kSweepThreads, 0, s>>>(d, n); }
        else { kJacobi<false><<<n, kSweepThreads, 0, s>>>(d, n); }
    }
    void launchSolve(hipStream_t s, const Dev& d, uint32_t held)
    {
        if (!d.nF) { return; }
        if (d.fastPairs) { kSolve<true><<<blocksOf(d.nF), kSweepThreads, 0, s>>>(d, held); }
        else { kSolve<false><<<blocksOf(d.nF), kSweepThreads, 0, s>>>(d, held); }
    }
    void launchFinalize(hipStream_t s, const Dev& d)
    {
        if (d.nF && d.nScenes) { kFinalize<<<d.nScenes, kSweepThreads, 0, s>>>(d, blocksOf(d.nF)); }
    }
    void launchIntegration(hipStream_t s, const Dev& d) { if (d.nF) { kIntegration<<<blocksOf(d.nF), kBlock, 0, s>>>(d); } }

    void launchRigidUpdate(hipStream_t s, const Dev& d, bool predicted) { if (d.nR) { kRigidUpdate<<<blocksOf(d.nR), kBlock, 0, s>>>(d, predicted); } }
    void launchRigidForces(hipStream_t s, const Dev& d, bool pressure)
    {
        if (d.nR) { kRigidForces<<<blocksOf(64ull * d.nR), kBlock, 0, s>>>(d, pressure); }
    }
    static void launchRigidBody(hipStream_t s, const Dev& d, uint32_t parts)
    {
        if (!d.nRB) { return; }
        const bool alone = d.mostR > kBodyParticles;
        constexpr uint32_t kUpdates = kBodyUpdate | kBodyUpdatePredicted;
        kRigidBody<<<d.nRB, kBodyThreads, 0, s>>>(d, alone ? parts & ~kUpdates : parts);
        if (alone && (parts & kUpdates)) { launchRigidUpdate(s, d, (parts & kBodyUpdatePredicted) != 0u); }
    }
    // the bodies after the non-pressure reaction: forces, prediction, predicted particles
    void launchRigidPredict(hipStream_t s, const Dev& d) { launchRigidBody(s, d, kBodySums | kBodyPredict | kBodyUpdatePredicted); }
    // after the pressure reaction: forces; then (a contact solve adds its loads between) the bodies' new state
    void launchRigidSums(hipStream_t s, const Dev& d) { launchRigidBody(s, d, kBodySums); }
    void launchRigidFinish(hipStream_t s, const Dev& d, bool sums)
    {
        launchRigidBody(s, d, (sums ? kBodySums : 0u) | kBodyPredict | kBodyIntegrate | kBodyUpdate);
    }
}
