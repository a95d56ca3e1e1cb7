// The drain of the path pools: how the last paths of a launch are saved, and traced to their end by groups of lanes. Used
// by the single-frame pool (path_pool.hpp) and the batched queue (batch.hip).
#pragma once

#include <type_traits>

#include "path_tracer.hpp"

namespace crvpt {

// ------------------------------------------------------------------------------------------------------------
// Drain
//
// A launch ends with its longest paths: once the claim queue is empty, waves run on with fewer and fewer live lanes, and
// a path's steps are a serial chain of a random block, a cell read and a density tap (about 0.8 us a step for a wave
// alone on its SIMD). Measured on the pool alone: a 64 x 64 frame of one sample is 0.5 ms of a 600-step chain; a
// 1280 x 720 one-sample frame empties its queue at 0.12 ms of 1.2 ms, the dense 128^3 next-event workload at
// 256^2 x 64 spp at 12.1 ms of 26.6 ms (chains of 13 000 steps). So a wave of the pool ends when its queue is empty and
// saves its live paths, and k_pathDrain spreads the saved paths over the chip and, as they finish, gives each path a
// group of lanes that looks up to kDrainGroup steps ahead (coopStep): the random numbers of a step depend on its index
// alone, and the next tentative collisions of a free path on nothing but them, so the group's lanes evaluate the steps'
// random blocks and density taps side by side and only the decisions follow in order. Every path makes the same steps
// with the same operations as in the pool, and they have to round alike: when a wave hands a path over depends on the
// schedule. Where the compiler's own choice of fused multiply-adds differs between the kernels the operation is written
// out (DenseAccessT::lookupWorldJ, cloudFiniteDifference); the tests compare whole images bit for bit.
// Kernel times in ms, pool alone -> pool and drain, for 100^2 x 1, 512^2 x 1, 1024^2 x 1, x 4 and x 16 samples:
//   dense 128^3, delta         0.86 -> 0.42   1.06 -> 0.81   1.73 -> 1.25   3.27 -> 2.60   8.84 -> 8.29
//   dense 128^3, next-event    7.40 -> 3.23   10.6 -> 6.44   14.0 -> 9.61   22.9 -> 18.8
//   sparse 512^3, ratio        1.80 -> 0.80   2.32 -> 1.32   3.22 -> 1.84   4.93 -> 3.55   12.1 -> 10.9
//   sparse 512^3, decomp.      0.61 -> 0.33   0.84 -> 0.60   1.11 -> 0.91   2.12 -> 1.94   5.95 -> 5.90
//   sparse 512^3, res. ratio   2.10 -> 1.27   2.45 -> 2.22   3.60 -> 3.22   7.87 -> 7.56   24.9 -> 25.2
// ------------------------------------------------------------------------------------------------------------
// Estimators with a drain (poolDrains, by mode): the spectral trackers' collision decisions change the path's weights at
// every step, so their next steps cannot be looked at ahead.
template <int MODE>
constexpr bool drains() {
    return !isSpectral<MODE>();
}

// Calls f on every 32-bit word of a path's state that MODE uses (pixel and frame follow from the unit, the constant
// fields from the start of the path).
template <int MODE, class F>
CRVPT_DEV void eachWord(PathState& st, Walker& W, F&& f) {
    auto v = [&](V3& a) {
        f(a.x);
        f(a.y);
        f(a.z);
    };
    f(st.unit);
    f(st.step);
    f(st.events);
    f(st.flags);
    v(W.o);
    v(W.w);
    f(W.t);
    f(W.tEnd);
    f(W.ix);
    f(W.iy);
    f(W.iz);
    f(W.nx);
    f(W.ny);
    f(W.nz);
    f(W.mu);
    f(W.tau);
    if (walksReferenceTable<MODE>()) f(W.muC);
    if (MODE == VPT_RESIDUAL_RATIO_TRACKING) {
        f(W.ctrl);
        f(st.wSum);
        f(st.resT);
        f(st.resDist);
    }
    if (MODE == VPT_RATIO_TRACKING || MODE == VPT_RESIDUAL_RATIO_TRACKING || isNee<MODE>()) f(st.thr);
    if (MODE == VPT_RESIDUAL_RATIO_TRACKING || isNee<MODE>()) v(st.color);
    if (isNee<MODE>()) {
        v(st.shadowScale);
        v(st.mainX);
        v(st.mainW);
    }
    if (MODE != VPT_RESIDUAL_RATIO_TRACKING && MODE != VPT_DECOMPOSITION_TRACKING) f(st.pendRho);
}

template <class T>
CRVPT_DEV uint32_t asWord(T v) {
    return __builtin_bit_cast(uint32_t, v);
}

// The wave's live lanes append their states to the queue: one record per path, so that the stores share one address
// (a word-major queue needs an address per word, and the registers for them made the pool spill in its loop). tag: a
// word of the caller's, kept behind the state where it is not 0.
template <int MODE>
CRVPT_DEV void saveState(PathState& st, Walker& W, const DrainQueue& Q, uint64_t alive, int lane, uint32_t tag) {
    uint32_t base = 0;
    if (lane == 0) base = atomicAdd(Q.count, uint32_t(__popcll(alive)));
    base = __builtin_amdgcn_readfirstlane(base);
    if (!(st.flags & PF_ALIVE)) return;
    uint32_t* p = Q.words + size_t(base + uint32_t(__popcll(alive & ((1ull << lane) - 1ull)))) * kDrainWords;
    int k = 0;
    eachWord<MODE>(st, W, [&](auto& w) { p[k++] = asWord(w); });
    if (tag != 0u) p[kDrainWords - 1] = tag;
}

// Lanes a path gets at most in the drain, as a power of two (1 / 4 / 8 / 16 / 32 lanes: 64 x 64 frame 0.60 / 0.45 / 0.38 /
// 0.42 / 0.53 ms, next-event workload 25.9 / 23.6 / 22.3 / 21.7 / 21.7 ms, delta sparse 5.81 / 5.60 / 5.60 / 5.75 / - ms);
// share (of 64) of the live lanes whose events a wave resolves together, steps between two looks at the live paths
// (both within 2 % from half to twice these), and the waves per SIMD the kernel is compiled for (3 / 4 / 5: next-event
// workload 26.1 / 23.0 / 23.6 ms).
constexpr int kDrainGroupLog = 3;
constexpr int kDrainResolve = 16;
constexpr int kDrainSteps = 8;
constexpr int kDrainWaves = 4;

// Up to 2^lg steps of a live path, by the 2^lg lanes from `base` on that all hold its state: lane base + sub evaluates
// the random block and the density tap of step st.step + sub. Returns false when the path finished.
template <int MODE, class Grid>
CRVPT_DEV bool coopStep(PathState& st, Walker& W, const SceneParams& P, const SupervoxelGrid& S, const Grid& grid,
                        typename Grid::Cache& gc, float4* feat, int lg, int sub, int base) {
    const int G = 1 << lg;
    const uint4 r = pathBlock(P, st, st.step + uint32_t(sub));
    const float e = __builtin_amdgcn_logf(uOpen(r.x)) * -0.693147182f;
    // the walk: every lane of the group makes all steps, and keeps what its own one ended at
    int ev = -1, last = 0;  // event of this lane's step (-1: behind the segment's end), last step walked
    float t = 0.0f, mu = 0.0f, muC = 0.0f, ctrl = 0.0f;
    for (int j = 0; j < G; j++) {
        const int evj = walkAdvance<MODE>(W, P, S, __shfl(e, base + j));
        if (j == sub) {
            ev = evj;
            t = W.t;
            mu = W.mu;
            muC = W.muC;
            ctrl = W.ctrl;
        }
        last = j;
        if (MODE == VPT_RESIDUAL_RATIO_TRACKING && evj != WALK_MOVED) W.ctrl = 0.0f;
        if (evj == WALK_END) break;
    }
    const float xi = u01(r.w);
    const bool control = MODE == VPT_DECOMPOSITION_TRACKING && xi * mu < muC;
    const bool collide = ev == WALK_COLLIDE;
    float rho = 0.0f;
    if (collide && !control) rho = tapDensity<MODE>(grid, P, W.o + W.w * t, r, gc);
    const uint64_t group = (~0ull >> (64 - G)) << base;
    if (MODE == VPT_RESIDUAL_RATIO_TRACKING) {
        const float factor = 1.0f - (P.extinction * rho - muC) * rcpf(mu);
        for (int j = 0; j <= last; j++) {
            const int evj = __shfl(ev, base + j);
            if (evj == WALK_MOVED) continue;
            st.thr *= __expf(-__shfl(ctrl, base + j));  // control transmittance of the walked stretch
            if (evj == WALK_END) {
                st.flags |= PF_PENDING | PF_PEND_END;
                break;
            }
            st.thr *= __shfl(factor, base + j);
            st.wSum += st.thr;
            if (__shfl(xi, base + j) * st.wSum < st.thr) {
                st.resT = st.thr;
                st.resDist = __shfl(t, base + j);
            }
        }
        st.step += uint32_t(last) + 1u;
        return true;
    }
    const float pReal = P.extinction * rho * rcpf(mu);
    if (isNee<MODE>() && (st.flags & PF_SHADOW)) {
        // ratio tracking (NeeTransmittance.glsl:107-113): a factor per collision, in order; 0 ends the ray
        const float factor = collide ? 1.0f - pReal : 1.0f;
        const bool ended = (__ballot(ev == WALK_END) & group) != 0ull;
        int stop = last;
        float f = __shfl(factor, base);
        for (int j = 0; j <= last; j++) {
            const float fn = __shfl(factor, base + ((j + 1) & (G - 1)));
            st.thr *= f;
            if (st.thr == 0.0f) {
                stop = j;
                break;
            }
            f = fn;
        }
        if (ended || st.thr == 0.0f) st.flags |= PF_PENDING | PF_PEND_END;
        st.step += uint32_t(stop) + 1u;
        return true;
    }
    // the first step that ends the free flight: a real collision, or the segment's end
    const bool real =
        collide && (MODE == VPT_DECOMPOSITION_TRACKING ? control || xi * mu < P.extinction * rho : xi < pReal);
    const uint64_t stops = __ballot(real || ev == WALK_END) & group;
    if (stops == 0ull) {
        st.step += uint32_t(last) + 1u;
        return true;
    }
    const int at = __builtin_ctzll(stops);
    st.step += uint32_t(at - base) + 1u;
    if (__shfl(ev, at) == WALK_END) {
        st.flags |= PF_PENDING | PF_PEND_END;
        return true;
    }
    W.t = __shfl(t, at);  // the walk restarts at the collision: nothing else of it is used
    const float xiAt = __shfl(xi, at), rhoAt = __shfl(rho, at), pRealAt = __shfl(pReal, at);
    const bool bounceLimit = P.maxBounces != 0u && (st.flags >> kBounceShift) >= P.maxBounces;
    if (MODE == VPT_DECOMPOSITION_TRACKING) {
        if (bounceLimit) {
            finishPath(st, v3(0.0f), true);
            return false;
        }
        st.pendRho = 0.0f;
        st.flags |= PF_PENDING;
        return true;
    }
    const bool absorbed = MODE != VPT_RATIO_TRACKING && xiAt < P.absorption * pRealAt;
    if (absorbed || bounceLimit) {
        if (absorbed)
            recordFirst<MODE, false>(st, P, grid, feat, W.o + W.w * W.t, isNee<MODE>() ? W.w : v3(0.0f), 0.0f,
                              rhoAt * (isNee<MODE>() ? P.extinctionMax : P.extinction), W.t);
        finishPath(st, isNee<MODE>() ? st.color : v3(0.0f), true);
        return false;
    }
    st.pendRho = rhoAt;
    st.flags |= PF_PENDING;
    return true;
}

// Traces the saved paths to their end. A wave owns a contiguous part of the queue: while it has paths to hand out, each
// lane walks one of its own; then the live paths are gathered and get groups of lanes. Path: what a path belongs to
// (k_pathDrain, k_batchDrain).
template <int MODE, class Path>
CRVPT_DEV void drainPaths(const DrainQueue& Q, Path& path) {
    const int lane = __lane_id();
    const uint32_t waves = gridDim.x * 4u;
    const uint32_t wave = blockIdx.x * 4u + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t total = *Q.count;
    uint32_t next = uint32_t(uint64_t(total) * wave / waves);
    const uint32_t end = uint32_t(uint64_t(total) * (wave + 1u) / waves);
    int lg = 0;
    PathState st;
    st.flags = 0;
    st.unit = st.pix = st.frame = st.step = st.events = st.taps = 0;
    st.thr = 1.0f;
    st.color = v3(0.0f);
    st.weights = v3(1.0f);
    st.pendRho = 0.0f;
    Walker W{};
    while (true) {
        uint64_t alive = __ballot((st.flags & PF_ALIVE) != 0);
        if (next < end) {  // one lane per path
            const uint32_t i = next + uint32_t(__popcll(~alive & ((1ull << lane) - 1ull)));
            if (!(st.flags & PF_ALIVE) && i < end) {
                const uint32_t* p = Q.words + size_t(i) * kDrainWords;
                int k = 0;
                eachWord<MODE>(st, W, [&](auto& w) {
                    w = __builtin_bit_cast(typename std::remove_reference<decltype(w)>::type, p[k++]);
                });
                path.open(st, p);
                W.ext = path.extinction();
            }
            next = min(end, next + uint32_t(__popcll(~alive)));
            alive = __ballot((st.flags & PF_ALIVE) != 0);
        }
        if (alive == 0ull) {
            if (next >= end) break;
            continue;
        }
        if (next >= end) {
            int want = lg;
            const int paths = __popcll(alive) >> lg;
            while (want < kDrainGroupLog && (paths << (want + 1)) <= 64) want++;
            if (want != lg) {
                // path k of the live ones goes to lanes k * 2^want ...
                uint64_t leaders = __ballot((st.flags & PF_ALIVE) != 0 && (lane & ((1 << lg) - 1)) == 0);
                int src = -1;
                for (int k = 0; leaders != 0ull; k++, leaders &= leaders - 1ull)
                    if (k == (lane >> want)) src = __builtin_ctzll(leaders);
                const int from = src < 0 ? lane : src;
                eachWord<MODE>(st, W, [&](auto& w) { w = __shfl(w, from); });
                st.pix = __shfl(st.pix, from);
                st.frame = __shfl(st.frame, from);
                path.moveFrom(from);
                if (src < 0) st.flags = 0;
                lg = want;
                alive = __ballot((st.flags & PF_ALIVE) != 0);
            }
        }
        const int sub = lane & ((1 << lg) - 1), base = lane - sub;
        const int resolveAt = max(1, (__popcll(alive) * kDrainResolve) >> 6);
        for (int k = 0; k < kDrainSteps; k++) {
            if ((st.flags & (PF_ALIVE | PF_PENDING)) == PF_ALIVE) {
                if (!path.step(st, W, lg, sub, base)) {
                    if (sub == 0) path.finish(st);
                    st.flags = 0;
                }
            }
            const uint64_t pend = __ballot((st.flags & PF_PENDING) != 0);
            if (pend != 0ull && (__popcll(pend) >= resolveAt || k == kDrainSteps - 1)) {
                if (st.flags & PF_PENDING) {
                    if (!path.resolve(st, W)) {
                        if (sub == 0) path.finish(st);
                        st.flags = 0;
                    }
                }
            }
        }
    }
}

}  // namespace crvpt
