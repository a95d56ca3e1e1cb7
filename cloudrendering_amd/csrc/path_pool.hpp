// Path pool kernels of the single-frame renderer (one translation unit per grid access variant, pool_*.hip).
//
// Work decomposition: a "unit" is one camera path (pixel p, sample s) with record slot s * (W*H) + p. Claims walk
// the image in 16 x 16 screen tiles, all of a launch's samples of one tile before the next, so a wave's 64
// consecutive claims are 64 neighbouring pixels of one sample (coherent primary rays) and the paths in flight read a
// small region of the volume. A persistent grid of waves drains a global claim counter: whenever lanes of a wave have no live path, one lane claims as many units as the
// wave has free lanes (ballot + popcount + one atomic) and the free lanes take them in lane order (mbcnt), so
// lanes refill at any step instead of idling until the longest path of the wave ends. Each path writes its
// radiance to its own slot; a separate kernel sums the slots of a pixel in sample order, so images are
// bit-reproducible whatever the lane/wave schedule was.
//
// Free-flight sampling walks a supervoxel majorant grid (piecewise-constant majorant along the ray): an Exp(1)
// optical budget is spent supervoxel by supervoxel, empty supervoxels cost one DDA step and no density fetch, and
// a tentative collision is accepted with probability sigma*rho / mu_local. With the grid disabled the walker
// degenerates to the reference's global majorant (extinction.x), i.e. the reference trackers' exact free-path
// distribution.
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "path_drain.hpp"

namespace crvpt {

#ifndef CRVPT_CLAIM_TILE
#define CRVPT_CLAIM_TILE 16
#endif
// Claims walk the image in square screen tiles of this edge, all of a launch's samples of one tile before the next
// (0: sample-major over the whole image). The paths in flight then cover a few tiles instead of a quarter of the
// image, so the volume region they read is small enough to stay in the L2 / Infinity Cache.
constexpr uint32_t kClaimTile = CRVPT_CLAIM_TILE;

CRVPT_DEV uint32_t claimCount(const SceneParams& P) {
    if (kClaimTile == 0u) return uint32_t(P.numUnits);
    const uint32_t tx = (uint32_t(P.width) + kClaimTile - 1u) / kClaimTile;
    const uint32_t ty = (uint32_t(P.height) + kClaimTile - 1u) / kClaimTile;
    return tx * ty * kClaimTile * kClaimTile * P.numFrames;
}

// Claim index -> launch slot sample * W*H + pixel (the record index); false for padding claims outside the image.
CRVPT_DEV bool claimToSlot(const SceneParams& P, uint32_t c, uint32_t& slot) {
    if (kClaimTile == 0u) {
        slot = c;
        return true;
    }
    constexpr uint32_t tp = kClaimTile * kClaimTile;
    const uint32_t w = uint32_t(P.width), h = uint32_t(P.height);
    const uint32_t tx = (w + kClaimTile - 1u) / kClaimTile;
    const uint32_t perTile = tp * P.numFrames;
    const uint32_t tile = udiv31(c, P.divTileClaims), rem = c - tile * perTile;
    const uint32_t s = rem / tp, q = rem - s * tp;
    const uint32_t ty = udiv31(tile, P.divTilesX);
    const uint32_t x = (tile - ty * tx) * kClaimTile + q % kClaimTile, y = ty * kClaimTile + q / kClaimTile;
    if (x >= w || y >= h) return false;
    slot = s * (w * h) + y * w + x;
    return true;
}

#ifndef CRVPT_CLAIM_PARTS
#define CRVPT_CLAIM_PARTS 32
#endif
// Claim partitions: the tiles are split into this many contiguous ranges, each with its own claim counter, and a
// workgroup first drains range blockIdx.x % parts, then the following ones. Workgroups are dispatched to the 8 XCDs
// round robin, so with a multiple of 8 ranges the paths in flight on one XCD come from a few bands of the image,
// which keeps the volume region they read, and so the XCD's L2 working set, small; the claims also spread over many
// counters instead of one.
constexpr uint32_t kClaimParts = CRVPT_CLAIM_PARTS;
#ifndef CRVPT_COUNTER_STRIDE
#define CRVPT_COUNTER_STRIDE 32
#endif
// Distance in 32-bit words between the claim counters of consecutive ranges (32: one 128-byte line each).
constexpr uint32_t kCounterStride = CRVPT_COUNTER_STRIDE;
// Word of the counters' buffer with the number of paths saved for the drain, behind the claim counters.
constexpr uint32_t kDrainCount = kClaimParts * kCounterStride;
constexpr uint32_t kClaimWords = kDrainCount + 1u;

CRVPT_DEV uint32_t partBegin(const SceneParams& P, uint32_t part) {
    if (kClaimParts == 1u) return part == 0u ? 0u : claimCount(P);
    const uint32_t tx = (uint32_t(P.width) + kClaimTile - 1u) / kClaimTile;
    const uint32_t ty = (uint32_t(P.height) + kClaimTile - 1u) / kClaimTile;
    const uint32_t tiles = tx * ty;
    return uint32_t(uint64_t(tiles) * part / kClaimParts) * (kClaimTile * kClaimTile * P.numFrames);
}

// STATS: instrumented variant that keeps the per-lane work counters and adds them to `stats` at exit; in the timed
// variant the counters are dead code and take no registers.
// DRAIN: the variant that leaves its last paths to k_pathDrain.
template <int MODE, class Grid, bool STATS, bool DRAIN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(poolWaves<MODE>()))) void k_pathPool(
        SceneParams P, Grid grid, SupervoxelGrid S, float4* __restrict__ out, uint32_t* __restrict__ counter,
        int stepsPerRefill, unsigned long long* __restrict__ stats, float4* __restrict__ feat, DrainQueue drain) {
    const int lane = __lane_id();
    PathState st;
    st.flags = 0;
    st.unit = 0;
    st.taps = 0;
    bool exhausted = false;
    uint32_t paths = 0;
    Walker W;
    W.svReads = 0;
    typename Grid::Cache gc;
    uint32_t part = kClaimParts == 1u ? 0u : blockIdx.x % kClaimParts;  // wave-uniform
    uint32_t partsLeft = kClaimParts;
    uint32_t begin = partBegin(P, part), count = partBegin(P, part + 1u) - begin;
    while (true) {
        // Refill until every lane holds a live path or the queue is drained: a claimed path whose camera ray misses
        // the volume finishes inside startPath, and its lane claims again before the wave steps.
        while (true) {
            const bool needs = !(st.flags & PF_ALIVE) && !exhausted;
            const uint64_t needMask = __ballot(needs);
            if (needMask == 0) break;
            const int leader = __ffsll((unsigned long long)needMask) - 1;
            const uint32_t want = uint32_t(__popcll(needMask));
            uint32_t base = 0;
            if (lane == leader) base = atomicAdd(&counter[part * kCounterStride], want);
            base = __builtin_amdgcn_readfirstlane(__shfl(base, leader));  // wave-uniform: the range state in SGPRs
            if (needs) {
                const uint32_t c = base + uint32_t(__popcll(needMask & ((1ull << lane) - 1ull)));
                if (c < count && claimToSlot(launchParams<MODE>(P), begin + c, st.unit)) {
                    paths++;
                    if (!startPath<MODE>(st, W, P, S, feat)) writePath(out, st);
                }
            }
            if (base + want >= count) {
                // this range is drained: the next one, until every range is
                if (--partsLeft == 0u) {
                    exhausted = true;
                } else {
                    part = part + 1u == kClaimParts ? 0u : part + 1u;
                    begin = partBegin(P, part);
                    count = partBegin(P, part + 1u) - begin;
                }
            }
        }
        // (the ballot in a variable of its own: tested in the conditions, the pool keeps 30 to 60 state words in scratch)
        const uint64_t alive = __ballot((st.flags & PF_ALIVE) != 0);
        if (alive == 0) break;                         // every lane is exhausted
        // The drain takes the live paths at once (waiting until at most 16, 32 or 48 lanes of a wave live: next-event
        // tracking of the dense 128^3 grid 8-33 % slower, 512^2 x 1 to 1920x1080 x 8, delta tracking 0-22 %).
        if (DRAIN && __ballot(exhausted) != 0) break;
        for (int k = 0; k < stepsPerRefill; k++) {
            if ((st.flags & (PF_ALIVE | PF_PENDING)) == PF_ALIVE) {
                if (!stepPath<MODE, Grid>(st, W, P, S, grid, gc, feat)) {
                    writePath(out, st);
                    st.flags = 0;
                }
            }
            const uint64_t pend = __ballot((st.flags & PF_PENDING) != 0);
            if (pend != 0ull && (__popcll(pend) >= kResolveLanes || k == stepsPerRefill - 1)) {
                if (st.flags & PF_PENDING) {
                    if (!resolvePending<MODE, Grid>(st, W, P, S, grid, feat)) {
                        writePath(out, st);
                        st.flags = 0;
                    }
                }
            }
        }
    }
    // behind the loop: inside it the state's addresses would be computed ahead and held in registers
    if (DRAIN) {
        const uint64_t alive = __ballot((st.flags & PF_ALIVE) != 0);
        if (alive != 0ull) saveState<MODE>(st, W, drain, alive, lane, 0u);
    }
    if (STATS) flushCounters(stats, st.taps, W.svReads, paths, gc.descents());
}

// Starts the camera paths of a small launch, a thread per claim, for the drain to trace from their beginning: such a
// launch needs no pool (a 64 x 64 frame spent 90 us in it, most of that on the 32 claim counters: 400 us a pass, now
// 300). Bound by the latency of one path's start.
template <int MODE, class Grid>
__global__ __launch_bounds__(256) void k_pathStart(SceneParams P, SupervoxelGrid S, float4* __restrict__ out,
                                                   float4* __restrict__ feat, DrainQueue drain) {
    const int lane = __lane_id();
    const uint32_t c = blockIdx.x * 256u + threadIdx.x;
    PathState st;
    st.flags = 0;
    st.unit = 0;
    st.pendRho = 0.0f;
    Walker W{};
    if (c < claimCount(P) && claimToSlot(launchParams<MODE>(P), c, st.unit)) {
        if (!startPath<MODE>(st, W, P, S, feat)) {
            writePath(out, st);
            st.flags = 0;
        }
    }
    const uint64_t alive = __ballot((st.flags & PF_ALIVE) != 0);
    if (alive != 0ull) saveState<MODE>(st, W, drain, alive, lane, 0u);
}

// Traces the paths the pool saved to their end.
template <int MODE, class Grid>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kDrainWaves))) void k_pathDrain(
        SceneParams P, Grid grid, SupervoxelGrid S, float4* __restrict__ out, float4* __restrict__ feat,
        DrainQueue drain) {
    struct Frame {
        const SceneParams& P;
        const Grid& grid;
        const SupervoxelGrid& S;
        float4* out;
        float4* feat;
        typename Grid::Cache gc;
        CRVPT_DEV void open(PathState& st, const uint32_t*) {
            const uint32_t s = udiv31(st.unit, P.divPixels);
            st.pix = st.unit - s * (uint32_t(P.width) * uint32_t(P.height));
            st.frame = P.frameBase + s;
        }
        CRVPT_DEV void moveFrom(int) {}
        CRVPT_DEV float extinction() const { return P.extinction; }
        CRVPT_DEV bool step(PathState& st, Walker& W, int lg, int sub, int base) {
            return coopStep<MODE, Grid>(st, W, P, S, grid, gc, feat, lg, sub, base);
        }
        CRVPT_DEV bool resolve(PathState& st, Walker& W) {
            return resolvePending<MODE, Grid>(st, W, P, S, grid, feat);
        }
        CRVPT_DEV void finish(const PathState& st) { writePath(out, st); }
    } frame{P, grid, S, out, feat, {}};
    drainPaths<MODE>(drain, frame);
}

// ------------------------------------------------------------------------------------------------------------
// Launch
// ------------------------------------------------------------------------------------------------------------
template <int MODE, class Grid>
static void launchPool(const SceneParams& P, const Grid& g, const SupervoxelGrid& S, float4* paths, uint32_t* counter,
                       const LaunchConfig& cfg, unsigned long long* stats, float4* feat, hipStream_t stream) {
    const dim3 grid(cfg.numBlocks), block(256);
    const int steps = cfg.stepsPerRefill;
    const DrainQueue& Q = cfg.drain;
    if (stats) {
        hipLaunchKernelGGL((k_pathPool<MODE, Grid, true, false>), grid, block, 0, stream, P, g, S, paths, counter, steps,
                           stats, feat, Q);
        return;
    }
    if constexpr (drains<MODE>()) {
        if (Q.words) {
            if (cfg.startBlocks > 0)
                hipLaunchKernelGGL((k_pathStart<MODE, Grid>), dim3(cfg.startBlocks), block, 0, stream, P, S, paths, feat,
                                   Q);
            else
                hipLaunchKernelGGL((k_pathPool<MODE, Grid, false, true>), grid, block, 0, stream, P, g, S, paths,
                                   counter, steps, stats, feat, Q);
            hipLaunchKernelGGL((k_pathDrain<MODE, Grid>), dim3(cfg.drainBlocks), block, 0, stream, P, g, S, paths, feat,
                               Q);
            return;
        }
    }
    hipLaunchKernelGGL((k_pathPool<MODE, Grid, false, false>), grid, block, 0, stream, P, g, S, paths, counter, steps,
                       stats, feat, Q);
}

// Launches the pool (and its drain) of P's estimator over one grid access variant; the claim counters and the drain
// queue's count are cleared by the caller.
template <class Grid>
hipError_t launchPoolT(const SceneParams& P, const Grid& grid, const SupervoxelGrid& S, float4* paths, uint32_t* counter,
                       const LaunchConfig& cfg, unsigned long long* stats, float4* feat, hipStream_t stream) {
    switch (P.mode) {
        case VPT_RATIO_TRACKING:
            launchPool<VPT_RATIO_TRACKING>(P, grid, S, paths, counter, cfg, stats, feat, stream);
            break;
        case VPT_NEXT_EVENT_TRACKING:
            launchPool<VPT_NEXT_EVENT_TRACKING>(P, grid, S, paths, counter, cfg, stats, feat, stream);
            break;
        case VPT_SPECTRAL_DELTA_TRACKING:
            launchPool<VPT_SPECTRAL_DELTA_TRACKING>(P, grid, S, paths, counter, cfg, stats, feat, stream);
            break;
        case VPT_NEXT_EVENT_TRACKING_SPECTRAL:
            launchPool<VPT_NEXT_EVENT_TRACKING_SPECTRAL>(P, grid, S, paths, counter, cfg, stats, feat, stream);
            break;
        case VPT_DECOMPOSITION_TRACKING:
            launchPool<VPT_DECOMPOSITION_TRACKING>(P, grid, S, paths, counter, cfg, stats, feat, stream);
            break;
        case VPT_RESIDUAL_RATIO_TRACKING:
            launchPool<VPT_RESIDUAL_RATIO_TRACKING>(P, grid, S, paths, counter, cfg, stats, feat, stream);
            break;
        default: launchPool<VPT_DELTA_TRACKING>(P, grid, S, paths, counter, cfg, stats, feat, stream); break;
    }
    return hipGetLastError();
}

// The timed pool kernel of an estimator without feature maps (occupancy query).
template <class Grid>
const void* poolKernelT(int mode) {
    switch (mode) {
        case VPT_RATIO_TRACKING: return (const void*)k_pathPool<VPT_RATIO_TRACKING, Grid, false, false>;
        case VPT_NEXT_EVENT_TRACKING: return (const void*)k_pathPool<VPT_NEXT_EVENT_TRACKING, Grid, false, false>;
        case VPT_SPECTRAL_DELTA_TRACKING: return (const void*)k_pathPool<VPT_SPECTRAL_DELTA_TRACKING, Grid, false, false>;
        case VPT_NEXT_EVENT_TRACKING_SPECTRAL: return (const void*)k_pathPool<VPT_NEXT_EVENT_TRACKING_SPECTRAL, Grid, false, false>;
        case VPT_DECOMPOSITION_TRACKING: return (const void*)k_pathPool<VPT_DECOMPOSITION_TRACKING, Grid, false, false>;
        case VPT_RESIDUAL_RATIO_TRACKING: return (const void*)k_pathPool<VPT_RESIDUAL_RATIO_TRACKING, Grid, false, false>;
        default: return (const void*)k_pathPool<VPT_DELTA_TRACKING, Grid, false, false>;
    }
}

#define CRVPT_INSTANTIATE_POOL(GRID)                                                                                 \
    template hipError_t launchPoolT<GRID>(const SceneParams&, const GRID&, const SupervoxelGrid&, float4*, uint32_t*, \
                                          const LaunchConfig&, unsigned long long*, float4*, hipStream_t);           \
    template const void* poolKernelT<GRID>(int);

}  // namespace crvpt
