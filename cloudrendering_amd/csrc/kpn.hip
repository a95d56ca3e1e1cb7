// Kernel-prediction denoiser application kernels (modules/kpn_module/src/Kernel.cu, caller
// src/Denoiser/PyTorchDenoiser.cpp:410-443):
//   perPixelKernel  out[n, c, y, x] = sum over the K x K window of weights[n, k, y, x] * image[n, c, y + dy, x + dx],
//                   taps outside the output extent (min of image and weight sizes) skipped (Kernel.cu:38-83);
//   invIterBase     the sigmoid-gated blend of the low-resolution prediction, the previous frame and the
//                   high-frequency detail (Kernel.cu:137-186), with the reference's weight batch stride of
//                   K*K*H*W although the fused weights hold K*K + 3 channels per batch;
//   softmax         over the first K*K channels of the fused weights, per pixel (torch::softmax(l, 1)).
#include <hip/hip_runtime.h>

#include <mutex>
#include <type_traits>

#include "render_api.hpp"

namespace crvpt {

constexpr int kKpnMaxChannels = 4;

// Blend of one pixel and channel (Kernel.cu:160-180): lfW, hfW, prW are the sigmoid gates. The reference blends with a
// double literal: (1.0 - prev_weight) and the sum are evaluated in double.
__device__ __forceinline__ float blend(float xHi, float xLo, float pLo, float prev, float lfW, float hfW, float prW,
                                       bool usePrevious) {
    float lf = lfW * pLo + (1.0f - lfW) * xLo;
    if (usePrevious) lf = float(double(lf) * (1.0 - double(prW)) + double(prev * prW));
    return hfW * (xHi - xLo + lf) + (1.0f - hfW) * lf;
}
__device__ __forceinline__ float sigmoid(float v) { return 1.0f / (1.0f + expf(-v)); }

// The K x K apply with the filtered image staged in LDS: a workgroup takes 64 x ROWS output pixels, a wave whole rows
// of 64, so that the weight planes, each read once, are read in full lines with K * K loads in flight, and the taps
// come from LDS. INV_ITER: the staged image is the inverse iteration's blend, computed on the way in (1.33 times per
// pixel at 16 rows, K = 5), and the weights pass a softmax in registers; nothing goes through memory between the three
// steps. Bound by the weight planes (107 of 160 B per pixel at K = 5, C = 3). The operations and their order are those
// of the separate kernels below, which remain for other K and for outputs that overlap an input.
// 1024 x 1024, K = 5, C = 3: 197 us as three kernels (softmax 106, apply 69, blend 22), now 43.5 us (3.7 TB/s).
constexpr int kApplyW = 64;

struct ApplyArgs {
    const float *image, *weights;        // INV_ITER: hiX, fused weights
    const float *loPred, *loX, *prev;    // INV_ITER only
    float* out;
    int h, w, imgH, imgW, wH, wW, loH, loW;
    int Ct;                              // weight planes per image
    int usePrevious;
};

template <int K, int C, int ROWS, bool INV_ITER>
__global__ __launch_bounds__(256) void k_applyTile(ApplyArgs A) {
    constexpr int R = K / 2, TW = kApplyW + 2 * R, TH = ROWS + 2 * R;
    __shared__ float tile[C][TH * TW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = blockIdx.z;
    const int x0 = int(blockIdx.x) * kApplyW, y0 = int(blockIdx.y) * ROWS;
    const size_t wPlane = size_t(A.wW) * A.wH, iPlane = size_t(A.imgW) * A.imgH, loPlane = size_t(A.loW) * A.loH;
    const float* img = A.image + size_t(n) * C * iPlane;
    for (int i = threadIdx.x; i < TH * TW; i += 256) {
        const int y = y0 + i / TW - R, x = x0 + i % TW - R;
        float v[C];
#pragma unroll
        for (int c = 0; c < C; c++) v[c] = 0.0f;
        if (unsigned(y) < unsigned(A.h) && unsigned(x) < unsigned(A.w)) {
            const size_t hi = size_t(y) * A.imgW + x;
            if (!INV_ITER) {
#pragma unroll
                for (int c = 0; c < C; c++) v[c] = img[c * iPlane + hi];
            } else if (x / 2 < A.loW && y / 2 < A.loH) {
                // (outside the low-resolution image the reference leaves its zero-initialised result, Kernel.cu:240)
                // gates with the reference's stride of K*K planes per batch
                const float* g = A.weights + size_t(n) * wPlane * (K * K) + K * K * wPlane + size_t(y) * A.wW + x;
                const float lfW = sigmoid(g[0]), hfW = sigmoid(g[wPlane]), prW = sigmoid(g[2 * wPlane]);
                const size_t lo = size_t(n) * C * loPlane + size_t(y / 2) * A.loW + x / 2;
#pragma unroll
                for (int c = 0; c < C; c++)
                    v[c] = blend(img[c * iPlane + hi], A.loX[lo + c * loPlane], A.loPred[lo + c * loPlane],
                                 A.usePrevious ? A.prev[(size_t(n) * C + c) * iPlane + hi] : 0.0f, lfW, hfW, prW,
                                 A.usePrevious != 0);
            }
        }
#pragma unroll
        for (int c = 0; c < C; c++) tile[c][i] = v[c];
    }
    __syncthreads();
    const int x = x0 + lane;
    if (x >= A.w) return;
    const size_t outPlane = size_t(A.w) * A.h;
    for (int row = wave; row < ROWS; row += 4) {
        const int y = y0 + row;
        if (y >= A.h) break;
        const float* wp = A.weights + size_t(n) * A.Ct * wPlane + size_t(y) * A.wW + x;
        float wt[K * K];
#pragma unroll
        for (int k = 0; k < K * K; k++) wt[k] = wp[k * wPlane];
        if (INV_ITER) {
            float m = -3.402823466e38f;
#pragma unroll
            for (int k = 0; k < K * K; k++) m = fmaxf(m, wt[k]);
            float s = 0.0f;
#pragma unroll
            for (int k = 0; k < K * K; k++) {
                wt[k] = expf(wt[k] - m);
                s += wt[k];
            }
            const float inv = 1.0f / s;
#pragma unroll
            for (int k = 0; k < K * K; k++) wt[k] *= inv;
        }
        float acc[C];
#pragma unroll
        for (int c = 0; c < C; c++) acc[c] = 0.0f;
#pragma unroll
        for (int k = 0; k < K * K; k++) {
            const int dy = k / K - R, dx = k % K - R;
            // a tap outside the extent is skipped whatever its weight
            const bool in = unsigned(y + dy) < unsigned(A.h) && unsigned(x + dx) < unsigned(A.w);
            const float v = in ? wt[k] : 0.0f;
#pragma unroll
            for (int c = 0; c < C; c++) acc[c] += v * tile[c][(row + R + dy) * TW + lane + R + dx];
        }
        float* ob = A.out + size_t(n) * C * outPlane + size_t(y) * A.w + x;
#pragma unroll
        for (int c = 0; c < C; c++) ob[c * outPlane] = acc[c];
    }
}

__global__ void k_perPixelKernel(const float* __restrict__ image, const float* __restrict__ weights,
                                 float* __restrict__ out, int K, int h, int w, int imgH, int imgW, int wH, int wW,
                                 int C) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int n = blockIdx.z;
    if (x >= w || y >= h) return;
    float acc[kKpnMaxChannels] = {0.0f, 0.0f, 0.0f, 0.0f};
    const size_t wPlane = size_t(wW) * wH, iPlane = size_t(imgW) * imgH;
    const float* wb = weights + size_t(n) * wPlane * K * K;
    const float* ib = image + size_t(n) * iPlane * C;
    int k = 0;
    for (int dy = -K / 2; dy <= K / 2; dy++) {
        const int ky = y + dy;
        for (int dx = -K / 2; dx <= K / 2; dx++, k++) {
            const int kx = x + dx;
            if (kx < 0 || kx >= w || ky < 0 || ky >= h) continue;
            const float wt = wb[size_t(k) * wPlane + size_t(y) * wW + x];
#pragma unroll
            for (int c = 0; c < kKpnMaxChannels; c++)
                if (c < C) acc[c] += wt * ib[size_t(c) * iPlane + size_t(ky) * imgW + kx];
        }
    }
    float* ob = out + size_t(n) * size_t(w) * h * C;
#pragma unroll
    for (int c = 0; c < kKpnMaxChannels; c++)
        if (c < C) ob[size_t(c) * size_t(w) * h + size_t(y) * w + x] = acc[c];
}

__global__ void k_invIterBase(const float* __restrict__ hiX, const float* __restrict__ loPred,
                              const float* __restrict__ loX, const float* __restrict__ prev,
                              const float* __restrict__ weights, float* __restrict__ out, int usePrevious, int K, int h,
                              int w, int imgH, int imgW, int loH, int loW, int wH, int wW, int C) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int n = blockIdx.z;
    const int lx = x / 2, ly = y / 2;
    if (x >= w || y >= h) return;
    if (lx >= loW || ly >= loH) {
        // outside the low-resolution image the reference leaves its zero-initialised result (Kernel.cu:240)
        for (int c = 0; c < C; c++)
            out[size_t(n) * size_t(w) * h * C + size_t(c) * size_t(w) * h + size_t(y) * w + x] = 0.0f;
        return;
    }
    const int kd = K * K;
    const size_t wPlane = size_t(wW) * wH;
    const float* wb = weights + size_t(n) * wPlane * kd;  // the reference's stride (K*K planes per batch)
    const float lfW = sigmoid(wb[size_t(kd) * wPlane + size_t(y) * wW + x]);
    const float hfW = sigmoid(wb[size_t(kd + 1) * wPlane + size_t(y) * wW + x]);
    const float prW = sigmoid(wb[size_t(kd + 2) * wPlane + size_t(y) * wW + x]);
    for (int c = 0; c < C; c++) {
        const size_t hi = size_t(n) * size_t(imgW) * imgH * C + size_t(c) * size_t(imgW) * imgH + size_t(y) * imgW + x;
        const size_t lo = size_t(n) * size_t(loW) * loH * C + size_t(c) * size_t(loW) * loH + size_t(ly) * loW + lx;
        out[size_t(n) * size_t(w) * h * C + size_t(c) * size_t(w) * h + size_t(y) * w + x] =
            blend(hiX[hi], loX[lo], loPred[lo], usePrevious ? prev[hi] : 0.0f, lfW, hfW, prW, usePrevious != 0);
    }
}

// Softmax over channels [0, K*K) of a [N, Ct, H, W] tensor into a [N, K*K, H, W] tensor (max-subtracted).
__global__ void k_softmaxChannels(const float* __restrict__ in, float* __restrict__ out, int Ct, int kk, int H, int W) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x;
    const int y = blockIdx.y * blockDim.y + threadIdx.y;
    const int n = blockIdx.z;
    if (x >= W || y >= H) return;
    const size_t plane = size_t(W) * H, px = size_t(y) * W + x;
    const float* ib = in + size_t(n) * plane * Ct;
    float* ob = out + size_t(n) * plane * kk;
    float m = -3.402823466e38f;
    for (int k = 0; k < kk; k++) m = fmaxf(m, ib[size_t(k) * plane + px]);
    float s = 0.0f;
    for (int k = 0; k < kk; k++) s += expf(ib[size_t(k) * plane + px] - m);
    const float inv = 1.0f / s;
    for (int k = 0; k < kk; k++) ob[size_t(k) * plane + px] = expf(ib[size_t(k) * plane + px] - m) * inv;
}

// Whether n floats at a and m floats at b share memory.
static bool overlap(const float* a, size_t n, const float* b, size_t m) {
    const uintptr_t p = reinterpret_cast<uintptr_t>(a), q = reinterpret_cast<uintptr_t>(b);
    return a && b && p < q + m * sizeof(float) && q < p + n * sizeof(float);
}

// Launches k_applyTile for the sizes that have one: K of 3, 5 or 7 and grids within the launch limits. The output is
// written while other workgroups read the inputs, so an output that overlaps one is left to the separate kernels.
template <bool INV_ITER>
static bool launchApplyTile(const ApplyArgs& A, int N, int C, int K, hipStream_t stream) {
    const size_t img = size_t(N) * C * A.imgH * A.imgW, lo = size_t(N) * C * A.loH * A.loW;
    const size_t out = size_t(N) * C * A.h * A.w, wts = size_t(N) * A.Ct * A.wH * A.wW;
    if ((K != 3 && K != 5 && K != 7) || C < 1 || C > kKpnMaxChannels) return false;
    if (overlap(A.out, out, A.image, img) || overlap(A.out, out, A.weights, wts)) return false;
    if (INV_ITER && (overlap(A.out, out, A.loPred, lo) || overlap(A.out, out, A.loX, lo) ||
                     (A.usePrevious && overlap(A.out, out, A.prev, img))))
        return false;
    // 16 rows per workgroup reuse more of the staged image; 4 rows where 16 would leave the chip idle, below two
    // workgroups per CU. An inverse iteration with 16 / 4 rows, workgroups of 16 rows in brackets: 640x480 (300) 17.9 /
    // 16.4 us, 1024x512 (512) 21.0 / 21.2, 720x720 (540) 24.2 / 25.9, 1024x768 (768) 28.5 / 29.7, 1024x1024 (1024)
    // 37.6 / 36.9, 1920x1080 (2040) 75 / 87; the plain apply 17.6 / 16.9 (768), 22.3 / 21.5 (1024) and 44 / 47.5 (2040).
    const unsigned gx = unsigned((A.w + kApplyW - 1) / kApplyW);
    const bool tall = size_t(gx) * ((A.h + 15) / 16) * N >= 512;
    const int rows = tall ? 16 : 4;
    const dim3 grid(gx, unsigned((A.h + rows - 1) / rows), unsigned(N)), block(256);
    if (grid.y > 65535u || grid.z > 65535u) return false;
    auto go = [&](auto kTag, auto cTag) {
        constexpr int k = decltype(kTag)::value, c = decltype(cTag)::value;
        if (tall) hipLaunchKernelGGL((k_applyTile<k, c, 16, INV_ITER>), grid, block, 0, stream, A);
        else hipLaunchKernelGGL((k_applyTile<k, c, 4, INV_ITER>), grid, block, 0, stream, A);
    };
    auto channels = [&](auto kTag) {
        switch (C) {
            case 1: go(kTag, std::integral_constant<int, 1>()); break;
            case 2: go(kTag, std::integral_constant<int, 2>()); break;
            case 3: go(kTag, std::integral_constant<int, 3>()); break;
            default: go(kTag, std::integral_constant<int, 4>()); break;
        }
    };
    if (K == 3) channels(std::integral_constant<int, 3>());
    else if (K == 5) channels(std::integral_constant<int, 5>());
    else channels(std::integral_constant<int, 7>());
    return true;
}

hipError_t launchPerPixelKernel(const float* image, const float* weights, float* out, int N, int C, int imgH,
                                int imgW, int wH, int wW, int K, hipStream_t stream) {
    const int h = imgH < wH ? imgH : wH, w = imgW < wW ? imgW : wW;
    const ApplyArgs A{image, weights, nullptr, nullptr, nullptr, out, h, w, imgH, imgW, wH, wW, 0, 0, K * K, 0};
    if (launchApplyTile<false>(A, N, C, K, stream)) return hipGetLastError();
    const dim3 block(16, 16, 1), grid((w + 15) / 16, (h + 15) / 16, N);
    hipLaunchKernelGGL(k_perPixelKernel, grid, block, 0, stream, image, weights, out, K, h, w, imgH, imgW, wH, wW, C);
    return hipGetLastError();
}

hipError_t launchInvIterBase(const float* hiX, const float* loPred, const float* loX, const float* prev,
                             const float* weights, float* out, bool usePrevious, int N, int C, int imgH, int imgW,
                             int loH, int loW, int wH, int wW, int K, hipStream_t stream) {
    const int h = imgH < wH ? imgH : wH, w = imgW < wW ? imgW : wW;
    const dim3 block(16, 16, 1), grid((w + 15) / 16, (h + 15) / 16, N);
    hipLaunchKernelGGL(k_invIterBase, grid, block, 0, stream, hiX, loPred, loX, prev, weights, out, int(usePrevious),
                       K, h, w, imgH, imgW, loH, loW, wH, wW, C);
    return hipGetLastError();
}

hipError_t launchSoftmaxChannels(const float* in, float* out, int N, int Ct, int kk, int H, int W,
                                 hipStream_t stream) {
    const dim3 block(16, 16, 1), grid((W + 15) / 16, (H + 15) / 16, N);
    hipLaunchKernelGGL(k_softmaxChannels, grid, block, 0, stream, in, out, Ct, kk, H, W);
    return hipGetLastError();
}

bool launchInvIterFused(const float* hiX, const float* loPred, const float* loX, const float* prev,
                        const float* weights, float* out, bool usePrevious, int N, int C, int imgH, int imgW, int loH,
                        int loW, int Ct, int wH, int wW, int K, hipStream_t stream) {
    const int h = imgH < wH ? imgH : wH, w = imgW < wW ? imgW : wW;
    const ApplyArgs A{hiX, weights, loPred, loX, prev, out, h, w, imgH, imgW, wH, wW, loH, loW, Ct, int(usePrevious)};
    return launchApplyTile<true>(A, N, C, K, stream);
}

// ------------------------------------------------------------------------------------------------------------
// Inverse-iteration apply without allocation: the blended base image and the normalised weights live in this file's
// static device array instead of renderer-owned buffers. Each GPU holds its own copy of the array; its address on
// a device is taken once (hipGetSymbolAddress with that device current) and kept per device. Calls on one GPU share
// the array, so calls that overlap in time on one GPU race; every call overwrites the part it uses completely, so
// nothing needs clearing between calls.
// ------------------------------------------------------------------------------------------------------------
static __device__ __align__(256) float scratch[kKpnNoAllocScratchFloats];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratchMutex;
float* g_scratchPtr[kMaxScratchDevices] = {};
}  // namespace

hipError_t kpnScratchSetup(float** ptr) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratchMutex);
    if (!g_scratchPtr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratchPtr[dev] = static_cast<float*>(p);
    }
    if (ptr) *ptr = g_scratchPtr[dev];
    return hipSuccess;
}

hipError_t launchInvIterNoAlloc(const float* hiX, const float* loPred, const float* loX, const float* prev,
                                const float* weights, float* out, bool usePrevious, int N, int C, int imgH, int imgW,
                                int loH, int loW, int Ct, int wH, int wW, int K, hipStream_t stream) {
    float* base = nullptr;
    hipError_t e = kpnScratchSetup(&base);
    if (e != hipSuccess) return e;
    if (launchInvIterFused(hiX, loPred, loX, prev, weights, out, usePrevious, N, C, imgH, imgW, loH, loW, Ct, wH, wW, K,
                           stream))
        return hipGetLastError();
    const int h = imgH < wH ? imgH : wH, w = imgW < wW ? imgW : wW;
    float* soft = base + size_t(N) * C * h * w;
    e = launchInvIterBase(hiX, loPred, loX, prev, weights, base, usePrevious, N, C, imgH, imgW, loH, loW, wH, wW, K,
                          stream);
    if (e != hipSuccess) return e;
    e = launchSoftmaxChannels(weights, soft, N, Ct, K * K, wH, wW, stream);
    if (e != hipSuccess) return e;
    return launchPerPixelKernel(base, soft, out, N, C, h, w, wH, wW, K, stream);
}

}  // namespace crvpt
