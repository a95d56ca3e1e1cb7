// Batched transmittance queries: n_samples estimates per ray, their mean and second moment.
//
// A unit is one estimate, unit = ray * n_samples + sample; every estimate has its own random stream (ray, sample, seed),
// so it does not depend on which lane makes it. A wave owns a contiguous range of units and gives each of its lanes the
// next one as soon as the lane's estimate is finished (ratio and delta tracking, one walker event per step), so lanes do
// not wait for the longest ray of the wave, and with several samples the lanes of a wave walk the same few rays.
// One sample: the estimate is the result. More: the estimates are stored and k_transmittanceMean sums each ray's in
// sample order in FP64.
//
// Bound by the walker's chain of dependent loads and its arithmetic, as the path pool. 10^6 rays through the 512^3
// NanoVDB cloud, ratio tracking, one sample: 3.03 ms a call with a thread per ray (64-bit grid offsets, lanes idle until
// the wave's longest ray ends, samples one after another), now 1.28 ms; 1900 rays of 21 samples: 9.6 -> 0.55 ms.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "path_tracer.hpp"

namespace crvpt {

// Per-lane work counters of the transmittance estimators (density taps, supervoxel table reads).
struct WorkCount {
    uint32_t taps = 0;
    uint32_t svReads = 0;
};

CRVPT_DEV float signf(float v) { return v > 0.0f ? 1.0f : (v < 0.0f ? -1.0f : 0.0f); }
CRVPT_DEV float fractf(float v) { return v - floorf(v); }

CRVPT_DEV bool refInside(const SupervoxelGrid& S, int x, int y, int z) {
    return x >= 0 && y >= 0 && z >= 0 && x < S.refGrid[0] && y < S.refGrid[1] && z < S.refGrid[2];
}
CRVPT_DEV size_t refIndex(const SupervoxelGrid& S, int x, int y, int z) {
    return (size_t(z) * S.refGrid[1] + y) * S.refGrid[0] + x;
}
CRVPT_DEV V3 gridDims(const SceneParams& P) {
    return v3(P.worldToTex[0] * (P.boxMax[0] - P.boxMin[0]), P.worldToTex[1] * (P.boxMax[1] - P.boxMin[1]),
              P.worldToTex[2] * (P.boxMax[2] - P.boxMin[2]));
}

struct RefDda {
    int step[3];
    float tMax[3], tDelta[3];
    int idx[3];
};

CRVPT_DEV bool refDdaInit(const SceneParams& P, const SupervoxelGrid& S, V3 x, V3 w, float dTotal, RefDda& q) {
    const V3 dims = gridDims(P);
    const V3 boxDelta = v3(P.boxMax) - v3(P.boxMin);
    const V3 sp = (x - v3(P.boxMin)) / boxDelta * dims / v3(float(S.refSize));
    const V3 ep = (x + w * dTotal - v3(P.boxMin)) / boxDelta * dims / v3(float(S.refSize));
#pragma unroll
    for (int a = 0; a < 3; a++) {
        const float s0 = comp(sp, a), e0 = comp(ep, a);
        const int st = int(signf(e0 - s0));
        const float td = st != 0 ? fminf(float(st) / (e0 - s0), 1e7f) : 1e7f;
        q.step[a] = st;
        q.tDelta[a] = td;
        q.tMax[a] = st > 0 ? td * (1.0f - fractf(s0)) : td * fractf(s0);
        q.idx[a] = int(floorf(s0));
    }
    return !(q.step[0] == 0 && q.step[1] == 0 && q.step[2] == 0);
}

CRVPT_DEV void refDdaAdvance(RefDda& q) {
    int a;
    if (q.tMax[0] < q.tMax[1]) a = q.tMax[0] < q.tMax[2] ? 0 : 2;
    else a = q.tMax[1] < q.tMax[2] ? 1 : 2;
    q.idx[a] += q.step[a];
    q.tMax[a] += q.tDelta[a];
}

CRVPT_DEV void refSvBounds(const SceneParams& P, const SupervoxelGrid& S, const int idx[3], V3& mn, V3& mx) {
    const V3 dims = gridDims(P);
    const V3 boxDelta = v3(P.boxMax) - v3(P.boxMin);
    const V3 lo = v3(float(idx[0] * S.refSize), float(idx[1] * S.refSize), float(idx[2] * S.refSize));
    const V3 hi = lo + v3(float(S.refSize));
    mn = lo / dims * boxDelta + v3(P.boxMin);
    mx = hi / dims * boxDelta + v3(P.boxMin);
}

template <class Grid>
CRVPT_DEV float rrtEstimator(const SceneParams& P, const Grid& grid, Rng& rng, V3 x, V3 w, float dStart, float dEnd,
                             float T, float& wSum, float& resT, float& resDist, float muC, float muR,
                             WorkCount& wc, typename Grid::Cache& gc) {
    const float Tc = __expf(-muC * (dEnd - dStart));
    float Tr = 1.0f;
    float dist = dStart;
    while (true) {
        const float t = rng.exponential() / muR;
        x += w * t;
        dist += t;
        if (dist >= dEnd) break;
        const float rho = density(grid, P, rng, x, gc);
        wc.taps++;
        Tr *= 1.0f - (P.extinction * rho - muC) / muR;
        const float Tlocal = T * Tr * __expf(-muC * (dist - dStart));
        wSum += Tlocal;
        if (rng.uniform() < Tlocal / wSum) {
            resT = Tlocal;
            resDist = dist;
        }
    }
    return Tc * Tr;
}

template <class Grid>
CRVPT_DEV float transmittanceRrt(const SceneParams& P, const SupervoxelGrid& S, const Grid& grid, Rng& rng, V3 x,
                                 V3 w, float limit) {
    const V3 eps = v3(1e-6f);
    float tMinVal, tMaxVal;
    if (!rayBoxIntersect(v3(P.boxMin) + eps, v3(P.boxMax) - eps, x, w, tMinVal, tMaxVal)) return 1.0f;
    x += w * tMinVal;
    const V3 oldX = x;
    const float lim = limit - tMinVal;
    RefDda q;
    if (!refDdaInit(P, S, x, w, tMaxVal - tMinVal, q)) return 1.0f;
    float T = 1.0f, wSum = 0.0f, resT = 0.0f, resDist = 0.0f;
    WorkCount wc;
    typename Grid::Cache gc;
    while (refInside(S, q.idx[0], q.idx[1], q.idx[2])) {
        const size_t si = refIndex(S, q.idx[0], q.idx[1], q.idx[2]);
        const float muC = S.rrt[2 * si], muR = S.rrt[2 * si + 1];
        V3 mn, mx;
        refSvBounds(P, S, q.idx, mn, mx);
        float a = 0.0f, b = 0.0f;
        rayBoxIntersect(mn, mx, oldX, w, a, b);
        b = fminf(b, lim);
        if (b > a) T *= rrtEstimator(P, grid, rng, oldX + w * a, w, a, b, T, wSum, resT, resDist, muC, muR, wc, gc);
        refDdaAdvance(q);
    }
    return T;
}

template <class Grid>
CRVPT_DEV float transmittanceDecomposition(const SceneParams& P, const SupervoxelGrid& S, const Grid& grid, Rng& rng,
                                           V3 x, V3 w, float limit) {
    const V3 eps = v3(1e-6f);
    float tMinVal, tMaxVal;
    if (!rayBoxIntersect(v3(P.boxMin) + eps, v3(P.boxMax) - eps, x, w, tMinVal, tMaxVal)) return 1.0f;
    const V3 dims = gridDims(P);
    const V3 boxDelta = v3(P.boxMax) - v3(P.boxMin);
    const V3 svSize = v3(float(S.refSize)) * boxDelta / dims;
    x += w * tMinVal;
    float travelled = tMinVal;
    typename Grid::Cache gc;
    const V3 sp = (x - v3(P.boxMin)) / boxDelta * dims / v3(float(S.refSize));
    int ix = int(floorf(sp.x)), iy = int(floorf(sp.y)), iz = int(floorf(sp.z));
    while (refInside(S, ix, iy, iz)) {
        const V3 minP = v3(P.boxMin) + v3(float(ix), float(iy), float(iz)) * svSize;
        const V3 maxP = minP + svSize;
        float a = 0.0f, b = 0.0f;
        rayBoxIntersect(minP, maxP, x, w, a, b);
        const float dMax = b - a;
        x += w * a;
        travelled += a;
        const float remaining = limit - travelled;
        if (remaining <= 0.0f) break;
        const float dUse = fminf(dMax, remaining);
        const size_t si = refIndex(S, ix, iy, iz);
        const float mmMin = S.decomp[2 * si], mmMax = S.decomp[2 * si + 1];
        if (mmMax >= 1e-5f) {
            const float muC = fmaxf(0.0000000001f, P.extinction * mmMin);
            const float muR = fmaxf(0.0000000001f, P.extinction * mmMax - muC);
            const float tc = rng.exponential() / muC;
            float tr = 0.0f;
            while (true) {
                tr += rng.exponential() / muR;
                if (tc >= dUse && tr >= dUse) break;
                if (tc <= tr) return 0.0f;
                const float rho = density(grid, P, rng, x + w * tr, gc);
                if (rng.uniform() * muR < P.extinction * rho - muC) return 0.0f;
            }
        }
        if (dUse < dMax) break;
        x = x + w * dMax;
        travelled += dMax;
        const V3 cc = (minP + maxP) * 0.5f;
        V3 mov = x + w * 0.00001f - cc;
        const V3 sm = v3(signf(mov.x), signf(mov.y), signf(mov.z));
        mov = mov * sm;
        ix += ((mov.x >= mov.y && mov.x >= mov.z) ? 1 : 0) * int(sm.x);
        iy += ((mov.y >= mov.x && mov.y >= mov.z) ? 1 : 0) * int(sm.y);
        iz += ((mov.z >= mov.x && mov.z >= mov.y) ? 1 : 0) * int(sm.z);
    }
    return 1.0f;
}

// The wave's range of units and the lane claims in it.
struct UnitRange {
    uint32_t next, end;
    CRVPT_DEV UnitRange(uint32_t units) {
        const uint32_t waves = gridDim.x * (blockDim.x / 64u), 
                       wave = blockIdx.x * (blockDim.x / 64u) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64u);
        next = uint32_t(uint64_t(units) * wave / waves);
        end = uint32_t(uint64_t(units) * (wave + 1u) / waves);
    }
};

struct RayBatch {
    const float *o, *d, *tmax;
    int nRays, nSamples;   // samples per ray of the call
    int ray0, sample0;     // first ray and sample of this launch
    int rays, samples;     // rays and samples per ray of this launch
    uint32_t seed;
};

struct RayResult {
    float *mean, *m2;      // one sample per ray: the results
    float* records;        // more: [rays][samples] estimates
    CRVPT_DEV void store(const RayBatch& B, uint32_t unit, float T) const {
        if (records) {
            records[unit] = T;
            return;
        }
        const uint32_t i = uint32_t(B.ray0) + unit;
        mean[i] = T;
        if (m2) m2[i] = float(double(T) * T);
    }
};

// Ray and random stream of a unit.
CRVPT_DEV uint32_t openUnit(const RayBatch& B, uint32_t unit, Rng& rng, V3& x, V3& w, float& lim) {
    const uint32_t r = unit / uint32_t(B.samples), s = unit - r * uint32_t(B.samples);
    const size_t i = size_t(B.ray0) + r;
    x = v3(B.o[3 * i], B.o[3 * i + 1], B.o[3 * i + 2]);
    w = v3(B.d[3 * i], B.d[3 * i + 1], B.d[3 * i + 2]);
    lim = B.tmax ? B.tmax[i] : kInf;
    rng.init(uint32_t(i), uint32_t(B.sample0) + s, B.seed ^ 0x5bd1e995u);
    return unit;
}

// Ratio tracking (BINARY: delta tracking) of the wave's units, refilled every kRaySteps walker events.
constexpr int kRaySteps = 8;

template <class Grid, bool BINARY>
__global__ __launch_bounds__(256) void k_transmittanceWalk(SceneParams P, Grid grid, SupervoxelGrid S, RayBatch B,
                                                           RayResult out) {
    UnitRange range(uint32_t(B.rays) * uint32_t(B.samples));
    const int lane = __lane_id();
    Walker W;
    W.svReads = 0;
    Rng rng;
    typename Grid::Cache gc;
    float T = 1.0f;
    uint32_t unit = 0;
    bool alive = false;
    while (true) {
        // hand out units until every lane walks one or the range is empty (a ray that misses the box ends at once)
        while (range.next < range.end) {
            const uint64_t free = __ballot(!alive);
            if (free == 0ull) break;
            const uint32_t u = range.next + uint32_t(__popcll(free & ((1ull << lane) - 1ull)));
            if (!alive && u < range.end) {
                V3 x, w;
                float lim;
                unit = openUnit(B, u, rng, x, w, lim);
                T = 1.0f;
                alive = walkerStart<VPT_DELTA_TRACKING>(W, P, S, x, w, lim);
                if (!alive) out.store(B, unit, T);
            }
            range.next += min(uint32_t(__popcll(free)), range.end - range.next);
        }
        if (__ballot(alive) == 0ull) break;
        for (int k = 0; k < kRaySteps; k++) {
            if (!alive) continue;
            const int ev = walkStep(W, rng, P, S);
            if (ev == WALK_COLLIDE) {
                const float rho = density(grid, P, rng, W.o + W.w * W.t, gc);
                const float pReal = P.extinction * rho / W.mu;
                if (!BINARY) {
                    T *= 1.0f - pReal;
                } else if (rng.uniform() < pReal) {
                    T = 0.0f;
                    alive = false;
                }
            } else if (ev == WALK_END) {
                alive = false;
            }
            if (!alive) out.store(B, unit, T);
        }
    }
}

// Residual ratio and decomposition tracking (the reference's traversal): a unit at a time per lane.
template <class Grid, bool DECOMPOSITION>
__global__ __launch_bounds__(256) void k_transmittanceTable(SceneParams P, Grid grid, SupervoxelGrid S, RayBatch B,
                                                            RayResult out) {
    UnitRange range(uint32_t(B.rays) * uint32_t(B.samples));
    for (uint32_t u = range.next + __lane_id(); u < range.end; u += 64u) {
        Rng rng;
        V3 x, w;
        float lim;
        openUnit(B, u, rng, x, w, lim);
        out.store(B, u, DECOMPOSITION ? transmittanceDecomposition(P, S, grid, rng, x, w, lim)
                                      : transmittanceRrt(P, S, grid, rng, x, w, lim));
    }
}

// Sums of a launch's estimates per ray, in sample order; sums (null where every ray's samples are in one launch) carries
// them from one launch of a ray's samples to the next.
__global__ void k_transmittanceMean(const float* __restrict__ records, RayBatch B, double2* __restrict__ sums,
                                    float* __restrict__ mean, float* __restrict__ m2) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= B.rays) return;
    double s1 = 0.0, s2 = 0.0;
    if (B.sample0 > 0) {
        s1 = sums[r].x;
        s2 = sums[r].y;
    }
    for (int s = 0; s < B.samples; s++) {
        const float T = records[size_t(r) * B.samples + s];
        s1 += T;
        s2 += double(T) * T;
    }
    if (B.sample0 + B.samples < B.nSamples) {
        sums[r] = make_double2(s1, s2);
        return;
    }
    mean[B.ray0 + r] = float(s1 / B.nSamples);
    if (m2) m2[B.ray0 + r] = float(s2 / B.nSamples);
}

// Persistent workgroups: a lane per unit, up to six waves per SIMD or as many as fit (10^6 rays with 4 / 5 / 6 / 8
// waves where 7 fit: 1.38 / 1.34 / 1.28 / 1.58 ms; the eighth starts when another has ended).
template <class Grid, class Kernel>
static void launchUnits(Kernel kernel, const SceneParams& P, const Grid& grid, const SupervoxelGrid& S,
                        const RayBatch& B, const RayResult& out, int cuCount, hipStream_t stream) {
    int fit = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&fit, reinterpret_cast<const void*>(kernel), 256, 0) !=
            hipSuccess || fit < 1)
        fit = 4;
    const uint64_t units = uint64_t(B.rays) * uint64_t(B.samples);
    const uint64_t blocks = std::min<uint64_t>((units + 255) / 256, uint64_t(cuCount) * uint64_t(std::min(fit, 6)));
    hipLaunchKernelGGL(kernel, dim3(unsigned(blocks)), dim3(256), 0, stream, P, grid, S, B, out);
}

template <class Grid>
static void launchWalk(const SceneParams& P, const Grid& grid, const SupervoxelGrid& S, int estimator,
                       const RayBatch& B, const RayResult& out, int cuCount, hipStream_t stream) {
    switch (estimator) {
        case T_RATIO: launchUnits(k_transmittanceWalk<Grid, false>, P, grid, S, B, out, cuCount, stream); break;
        case T_RESIDUAL_RATIO: launchUnits(k_transmittanceTable<Grid, false>, P, grid, S, B, out, cuCount, stream); break;
        case T_DECOMPOSITION: launchUnits(k_transmittanceTable<Grid, true>, P, grid, S, B, out, cuCount, stream); break;
        default: launchUnits(k_transmittanceWalk<Grid, true>, P, grid, S, B, out, cuCount, stream); break;
    }
}

hipError_t launchTransmittance(const SceneParams& P, const DenseGrid* dense, const NanoGrid* nano,
                               const SupervoxelGrid& S, int estimator, const float* o, const float* d,
                               const float* tmax, int nRays, int nSamples, uint32_t seed, float* mean, float* m2,
                               const TransmittancePlan& plan, void* work, int cuCount, hipStream_t stream) {
    const size_t samples = plan.samples, rays = plan.rays;
    double2* sums = plan.sumBytes > 0 ? reinterpret_cast<double2*>(work) : nullptr;
    float* records = plan.recordBytes > 0
                             ? reinterpret_cast<float*>(reinterpret_cast<char*>(work) + plan.sumBytes)
                             : nullptr;
    const RayResult out{mean, m2, records};
    const bool tri = P.interpolation == INTERP_TRILINEAR;
    for (size_t r0 = 0; r0 < size_t(nRays); r0 += rays)
        for (size_t s0 = 0; s0 < size_t(nSamples); s0 += samples) {
            RayBatch B{o, d, tmax, nRays, nSamples, int(r0), int(s0), int(std::min(rays, size_t(nRays) - r0)),
                       int(std::min(samples, size_t(nSamples) - s0)), seed};
            // the grid variants of the path kernels (launchRender); the trilinear code stays in the general ones
            if (nano && (nano->wide || !nano->tapDiag || tri))
                launchWalk(P, NanoAccess{*nano}, S, estimator, B, out, cuCount, stream);
            else if (nano)
                launchWalk(P, NanoAccessNarrowPoint{*nano}, S, estimator, B, out, cuCount, stream);
            else
                launchWalk(P, DenseAccess{*dense}, S, estimator, B, out, cuCount, stream);
            if (records)
                hipLaunchKernelGGL(k_transmittanceMean, dim3(unsigned((B.rays + 255) / 256)), dim3(256), 0, stream,
                                   records, B, sums, mean, m2);
            if (const hipError_t e = hipGetLastError()) return e;
        }
    return hipSuccess;
}

}  // namespace crvpt
