// Batched render queue: many requests of different volumes, resolutions and sample counts traced by one persistent
// launch (no reference counterpart; the reference renders one frame per call, Module.cpp:286-317).
//
// Work decomposition: request r owns the batch units [unitBegin_r, unitBegin_r + groups_r * W_r * H_r); unit
// unitBegin_r + g * (W_r*H_r) + p traces samples [g*G, min(spp_r, (g+1)*G)) of pixel p, one after another on the
// same lane, and leaves one record (the sum of its samples' radiance). The units of one group are neighbouring
// pixels, so a wave starts on coherent camera rays as in the single-frame pool. Lanes claim units exactly like the
// single-frame pool (ballot, one atomic per wave, lane rank by popcount); a lane whose unit has samples left starts
// the next one in place, without claiming. The request of a unit is found by binary search over the requests' first
// units; a lane reads its request's scene constants and volume through the device request table.
//
// Every path draws the same counter-based random numbers as in a single-frame render of the same request (pixel,
// frame number, seed offset) and runs the same device code, so a batch with G = 1 reproduces the single-frame images
// up to the last bits (the compiler forms fused multiply-adds differently in the two kernels); larger G also
// regroups the floating-point sum over samples.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "path_drain.hpp"

namespace crvpt {

// A request's volume, read through the device request table: dense or NanoVDB by P.sparse.
struct BatchGrid {
    const BatchRequest* R;
    using Cache = LeafCache;
    template <class TAP>
    CRVPT_DEV float lookupWorldJ(const SceneParams& P, V3 pos, float jx, float jy, float jz, LeafCache& c) const {
        if (R->P.sparse) return NanoAccess{R->nano}.lookupWorldJ(P, pos, jx, jy, jz, c);
        return DenseAccess{R->dense}.lookupWorldJ<TAP>(P, pos, jx, jy, jz);
    }
};
// Batches write no feature maps.
template <bool FUSE>
CRVPT_DEV V3 cloudFiniteDifference(const BatchGrid&, const SceneParams&, const PathState&, V3) { return v3(0.0f); }

// Last request r with begins[r] <= q (begins ascending, begins[0] = 0).
CRVPT_DEV int findRequest(const uint64_t* __restrict__ begins, int n, uint64_t q) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (begins[mid] <= q) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

#ifndef CRVPT_BATCH_CLAIM_PARTS
#define CRVPT_BATCH_CLAIM_PARTS 1
#endif
// Unit partitions: the batch's units can be split into this many contiguous ranges (consecutive requests), each with
// its own claim counter; a workgroup first drains range blockIdx.x % parts, then the following ones. One range (a
// single counter over all units) measured fastest on the 64-request workload (8 ranges: 4 % slower), so it is the
// default.
constexpr uint32_t kBatchParts = CRVPT_BATCH_CLAIM_PARTS;

CRVPT_DEV uint32_t unitPartBegin(uint32_t totalUnits, uint32_t part) {
    return uint32_t(uint64_t(totalUnits) * part / kBatchParts);
}

// DRAIN (units of one sample): the pool leaves its last paths to k_batchDrain.
template <int MODE, bool DRAIN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(batchPoolWaves<MODE>()))) void k_batchPool(
        const BatchRequest* __restrict__ reqs, const uint64_t* __restrict__ unitBegins, int nreq, uint32_t totalUnits,
        uint32_t samplesPerUnit, const uint32_t* __restrict__ frameOffset, float4* __restrict__ records,
        uint32_t* __restrict__ counter, int stepsPerRefill, DrainQueue drain) {
    const int lane = __lane_id();
    const uint32_t frameOff = *frameOffset;
    PathState st;
    st.flags = 0;
    st.unit = 0;
    st.pix = 0;
    st.taps = 0;
    int req = 0;
    uint32_t left = 0, sample = 0;
    V3 sum = v3(0.0f);
    bool exhausted = false;
    Walker W;
    W.svReads = 0;
    LeafCache gc;
    // A finished sample adds to its unit's sum; the unit's last sample stores the record.
    auto finishSample = [&]() {
        sum += st.color;
        st.flags = 0;
        if (left == 0u) records[st.unit] = make_float4(sum.x, sum.y, sum.z, 0.0f);
    };
    uint32_t part = kBatchParts == 1u ? 0u : blockIdx.x % kBatchParts;  // wave-uniform
    uint32_t partsLeft = kBatchParts;
    uint32_t begin = unitPartBegin(totalUnits, part), count = unitPartBegin(totalUnits, part + 1u) - begin;
    while (true) {
        while (true) {
            const bool claim = !(st.flags & PF_ALIVE) && left == 0u && !exhausted;
            const uint64_t claimMask = __ballot(claim);
            if (claimMask != 0ull) {
                const int leader = __ffsll((unsigned long long)claimMask) - 1;
                const uint32_t want = uint32_t(__popcll(claimMask));
                uint32_t base = 0;
                if (lane == leader) base = atomicAdd(&counter[part], want);
                base = __shfl(base, leader);
                const bool drained = base + want >= count;
                const uint32_t partStart = begin, partCount = count;
                if (drained) {
                    // this range is drained: the next one, until every range is
                    if (--partsLeft == 0u) {
                        exhausted = true;
                    } else {
                        part = part + 1u == kBatchParts ? 0u : part + 1u;
                        begin = unitPartBegin(totalUnits, part);
                        count = unitPartBegin(totalUnits, part + 1u) - begin;
                    }
                }
                if (claim) {
                    const uint32_t c = base + uint32_t(__popcll(claimMask & ((1ull << lane) - 1ull)));
                    const uint32_t u = partStart + c;
                    if (c < partCount) {
                        const int r = findRequest(unitBegins, nreq, u);
                        if (r != req) {
                            gc = LeafCache();  // the memo holds byte offsets into the previous request's grid
                            req = r;
                        }
                        const BatchRequest& R = reqs[req];
                        const uint32_t npix = uint32_t(R.P.width) * uint32_t(R.P.height);
                        const uint32_t local = u - uint32_t(unitBegins[req]);
                        const uint32_t g = local / npix;
                        st.unit = u;
                        st.pix = local - g * npix;
                        sample = g * samplesPerUnit;
                        left = min(samplesPerUnit, R.spp - sample);
                        sum = v3(0.0f);
                    }
                }
            }
            if (!(st.flags & PF_ALIVE) && left > 0u) {
                const BatchRequest& R = reqs[req];
                st.frame = R.P.frameBase + frameOff + sample;
                sample++;
                left--;
                if (!startPathAt<MODE>(st, W, R.P, R.S, nullptr, R.P.invViewProj)) finishSample();
            }
            if (__ballot(!(st.flags & PF_ALIVE) && (left > 0u || !exhausted)) == 0ull) break;
        }
        // (the ballot in a variable of its own, see k_pathPool)
        const uint64_t alive = __ballot((st.flags & PF_ALIVE) != 0);
        if (alive == 0ull) break;                         // every lane is exhausted
        if (DRAIN && __ballot(exhausted) != 0ull) break;  // the drain takes the live paths
        for (int k = 0; k < stepsPerRefill; k++) {
            if ((st.flags & (PF_ALIVE | PF_PENDING)) == PF_ALIVE) {
                const BatchRequest& R = reqs[req];
                if (!stepPath<MODE, BatchGrid>(st, W, R.P, R.S, BatchGrid{&R}, gc, nullptr)) finishSample();
            }
            const uint64_t pend = __ballot((st.flags & PF_PENDING) != 0);
            if (pend != 0ull && (__popcll(pend) >= kResolveLanes || k == stepsPerRefill - 1)) {
                if (st.flags & PF_PENDING) {
                    const BatchRequest& R = reqs[req];
                    if (!resolvePending<MODE, BatchGrid>(st, W, R.P, R.S, BatchGrid{&R}, nullptr)) finishSample();
                }
            }
        }
    }
    if (DRAIN) {
        const uint64_t alive = __ballot((st.flags & PF_ALIVE) != 0);
        if (alive != 0ull) saveState<MODE>(st, W, drain, alive, lane, uint32_t(req) + 1u);
    }
}

// Traces the paths the batch pool saved to their end; a path's request is the word behind its state.
template <int MODE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kDrainWaves))) void k_batchDrain(
        const BatchRequest* __restrict__ reqs, const uint64_t* __restrict__ unitBegins,
        const uint32_t* __restrict__ frameOffset, float4* __restrict__ records, DrainQueue drain) {
    struct Request {
        const BatchRequest* reqs;
        const uint64_t* unitBegins;
        uint32_t frameOff;
        float4* records;
        int req;
        LeafCache gc;
        CRVPT_DEV void open(PathState& st, const uint32_t* words) {
            const int r = int(words[kDrainWords - 1]) - 1;
            if (r != req) gc = LeafCache();  // the memo holds byte offsets into the previous request's grid
            req = r;
            const BatchRequest& R = reqs[req];
            const uint32_t npix = uint32_t(R.P.width) * uint32_t(R.P.height);
            const uint32_t local = st.unit - uint32_t(unitBegins[req]);
            const uint32_t sample = local / npix;  // a unit is one sample
            st.pix = local - sample * npix;
            st.frame = R.P.frameBase + frameOff + sample;
        }
        CRVPT_DEV void moveFrom(int from) {
            req = __shfl(req, from);
            gc = LeafCache();
        }
        CRVPT_DEV float extinction() const { return reqs[req].P.extinction; }
        CRVPT_DEV bool step(PathState& st, Walker& W, int lg, int sub, int base) {
            const BatchRequest& R = reqs[req];
            return coopStep<MODE, BatchGrid>(st, W, R.P, R.S, BatchGrid{&R}, gc, nullptr, lg, sub, base);
        }
        CRVPT_DEV bool resolve(PathState& st, Walker& W) {
            const BatchRequest& R = reqs[req];
            return resolvePending<MODE, BatchGrid>(st, W, R.P, R.S, BatchGrid{&R}, nullptr);
        }
        CRVPT_DEV void finish(const PathState& st) {
            records[st.unit] = make_float4(st.color.x, st.color.y, st.color.z, 0.0f);
        }
    } request{reqs, unitBegins, *frameOffset, records, 0, {}};
    drainPaths<MODE>(drain, request);
}

// Per pixel of every request: the sum of its units' records in group order, divided by spp (the single-frame
// accumulation's order and rounding when every unit holds one sample), written as [C, H, W] with alpha 1.
__global__ void k_batchResolve(const BatchRequest* __restrict__ reqs, const uint64_t* __restrict__ pixBegins,
                               int nreq, uint64_t totalPix, const float4* __restrict__ records) {
    const uint64_t q = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (q >= totalPix) return;
    const int r = findRequest(pixBegins, nreq, q);
    const BatchRequest& R = reqs[r];
    const uint32_t npix = uint32_t(R.P.width) * uint32_t(R.P.height);
    const uint32_t p = uint32_t(q - pixBegins[r]);
    // FP64 sums over the units (see k_accumulate: float sums of many equal samples drift)
    double sx = 0.0, sy = 0.0, sz = 0.0;
    for (uint32_t g = 0; g < R.groups; g++) {
        const float4 v = records[R.unitBegin + uint64_t(g) * npix + p];
        sx += double(v.x);
        sy += double(v.y);
        sz += double(v.z);
    }
    const double inv = 1.0 / double(R.spp);
    float* o = R.out;
    o[p] = float(sx * inv);
    o[npix + p] = float(sy * inv);
    o[2 * size_t(npix) + p] = float(sz * inv);
    if (R.channels == 4) o[3 * size_t(npix) + p] = 1.0f;
}

__global__ void k_setU32(uint32_t* p, uint32_t v) {
    if (threadIdx.x == 0) *p = v;
}

// Calls f with the estimator as an integral constant.
template <class F>
static void withMode(int mode, F&& f) {
    switch (mode) {
        case VPT_RATIO_TRACKING: f(std::integral_constant<int, VPT_RATIO_TRACKING>()); break;
        case VPT_NEXT_EVENT_TRACKING: f(std::integral_constant<int, VPT_NEXT_EVENT_TRACKING>()); break;
        case VPT_SPECTRAL_DELTA_TRACKING: f(std::integral_constant<int, VPT_SPECTRAL_DELTA_TRACKING>()); break;
        case VPT_NEXT_EVENT_TRACKING_SPECTRAL:
            f(std::integral_constant<int, VPT_NEXT_EVENT_TRACKING_SPECTRAL>());
            break;
        case VPT_DECOMPOSITION_TRACKING: f(std::integral_constant<int, VPT_DECOMPOSITION_TRACKING>()); break;
        case VPT_RESIDUAL_RATIO_TRACKING: f(std::integral_constant<int, VPT_RESIDUAL_RATIO_TRACKING>()); break;
        default: f(std::integral_constant<int, VPT_DELTA_TRACKING>()); break;
    }
}

int batchOccupancyBlocksPerCU(int mode, int blockSize) {
    const void* kernel = nullptr;
    withMode(mode, [&](auto m) { kernel = (const void*)k_batchPool<decltype(m)::value, false>; });
    int blocks = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, blockSize, 0);
    if (e != hipSuccess || blocks <= 0) return 1;
    return blocks;
}

hipError_t launchSetU32(uint32_t* p, uint32_t v, hipStream_t stream) {
    hipLaunchKernelGGL(k_setU32, dim3(1), dim3(64), 0, stream, p, v);
    return hipGetLastError();
}

hipError_t launchBatch(int mode, const BatchRequest* reqs, const uint64_t* unitBegins, const uint64_t* pixBegins,
                       int nreq, uint32_t totalUnits, uint64_t totalPix, const BatchLaunch& cfg,
                       const uint32_t* frameOffset, float4* records, uint32_t* counter, uint32_t* drainWords,
                       uint32_t drainBlocks, hipStream_t stream) {
    if (cfg.blockSize <= 0 || cfg.blockSize > 256 || cfg.blockSize % 64 != 0 || cfg.numBlocks == 0 ||
        cfg.samplesPerUnit == 0 || cfg.stepsPerRefill <= 0 || (drainWords && cfg.samplesPerUnit != 1u))
        return hipErrorInvalidValue;
    for (uint32_t p = 0; p < kBatchParts; p++) hipLaunchKernelGGL(k_setU32, dim3(1), dim3(64), 0, stream, counter + p, 0u);
    DrainQueue drain{drainWords, counter + kBatchParts};
    const dim3 grid(cfg.numBlocks), block(cfg.blockSize);
    if (drainWords) hipLaunchKernelGGL(k_setU32, dim3(1), dim3(64), 0, stream, drain.count, 0u);
    hipError_t e = hipSuccess;
    withMode(mode, [&](auto m) {
        constexpr int M = decltype(m)::value;
        if constexpr (drains<M>()) {
            if (drainWords) {
                hipLaunchKernelGGL((k_batchPool<M, true>), grid, block, 0, stream, reqs, unitBegins, nreq, totalUnits,
                                   cfg.samplesPerUnit, frameOffset, records, counter, cfg.stepsPerRefill, drain);
                e = hipGetLastError();
                if (e != hipSuccess) return;
                hipLaunchKernelGGL(k_batchDrain<M>, dim3(drainBlocks), dim3(256), 0, stream, reqs, unitBegins,
                                   frameOffset, records, drain);
                e = hipGetLastError();
                return;
            }
        }
        hipLaunchKernelGGL((k_batchPool<M, false>), grid, block, 0, stream, reqs, unitBegins, nreq, totalUnits,
                           cfg.samplesPerUnit, frameOffset, records, counter, cfg.stepsPerRefill, drain);
        e = hipGetLastError();
    });
    if (e != hipSuccess) return e;
    const uint64_t blocks = (totalPix + 255) / 256;
    hipLaunchKernelGGL(k_batchResolve, dim3(unsigned(blocks)), dim3(256), 0, stream, reqs, pixBegins, nreq, totalPix,
                       (const float4*)records);
    return hipGetLastError();
}

}  // namespace crvpt
