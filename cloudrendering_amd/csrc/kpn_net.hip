// Kernel-prediction denoiser network on gfx950: six 3x3 convolutions (15 -> 32 -> 32 -> 32 -> 32 -> 32 -> 25
// channels, ReLU between them) whose 25 output logits per pixel are turned by a softmax into a 5x5 filter applied to
// the noisy radiance (the per-pixel kernel of modules/kpn_module Kernel.cu:38-83 with the caller's softmax,
// PyTorchDenoiser.cpp:428-431). Training: relative-MSE loss against a high-sample target, hand-written backward
// passes and Adam.
//
// Layout: activations are NHWC bf16 with 32 channels per pixel (the 15 input features and the 25 logits are padded
// with zero channels), so one 3x3 tap of one pixel is exactly the K = 32 operand of v_mfma_f32_16x16x32_bf16.
// Convolutions are implicit GEMMs: a workgroup stages a 16x16 output tile plus its one-pixel halo in LDS; each of
// its four waves owns four rows of 16 pixels (four 16-pixel M tiles) and both 16-channel N tiles, and accumulates
// nine MFMAs (one per tap) per M/N tile pair in FP32. Weights are pre-swizzled into per-lane MFMA fragments (bf16)
// from FP32 master copies after every optimiser step.
//
// MFMA lane layout (16x16x32, bf16 in, f32 out): lane l supplies A[m = l % 16][k = 8 * (l / 16) + j] and
// B[k = 8 * (l / 16) + j][n = l % 16] for j < 8, and receives C[m = 4 * (l / 16) + i][n = l % 16] for i < 4.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "render_api.hpp"

namespace crvpt {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kC = kKpnChannels;  // 32 channels per activation pixel
constexpr int kTile = 16;         // output tile edge in pixels
constexpr int kHalo = kTile + 2;  // staged input tile edge (3x3 halo)
constexpr int kPixStride = 40;    // bf16 per staged pixel in LDS: 32 channels + 8 of padding (80 B, 16-B aligned)

enum : int { EPI_RELU_BF16 = 0, EPI_LINEAR_F32 = 1, EPI_MASK_BF16 = 2 };

__device__ __forceinline__ f32x4 mfma16(const bf16x8& a, const bf16x8& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Tile index of a persistent workgroup's k-th tile. Workgroups go to the 8 XCDs round robin, each with its own L2:
// XCD x takes the x-th eighth of the tiles, so that neighbouring tiles, which share their halo pixels, meet in one L2.
constexpr int kXcds = 8;

struct TileWalk {
    int tilesX, tilesY, end, step, ti;
    int n, y0, x0;
    __device__ __forceinline__ TileWalk(int N, int H, int W) {
        tilesX = (W + kTile - 1) / kTile;
        tilesY = (H + kTile - 1) / kTile;
        const int numTiles = N * tilesX * tilesY;
        const int xcd = int(blockIdx.x) % kXcds, slot = int(blockIdx.x) / kXcds;
        const int groups = min(int(gridDim.x), kXcds);  // XCDs that have a workgroup
        const int begin = int(int64_t(numTiles) * xcd / groups);
        end = int(int64_t(numTiles) * (xcd + 1) / groups);
        step = (int(gridDim.x) - xcd + kXcds - 1) / kXcds;  // workgroups of this XCD
        ti = begin + slot;
        locate();
    }
    __device__ __forceinline__ void locate() {
        n = ti / (tilesX * tilesY);
        const int r = ti - n * tilesX * tilesY;
        y0 = (r / tilesX) * kTile;
        x0 = (r % tilesX) * kTile;
    }
    __device__ __forceinline__ bool valid() const { return ti < end; }
    __device__ __forceinline__ void next() {
        ti += step;
        locate();
    }
};

// The (16 + 2)^2 input pixels of CIN channels (32, or 16 for the packed features) around output tile (y0, x0) of image
// n, zero outside the image, in 16-byte chunks of which thread t holds chunks t, t + THREADS, ... in registers between
// load() and store() into LDS (STRIDE bf16 per pixel). The next tile's halo is loaded before the current tile is computed, so its latency is
// hidden behind the MFMAs and stores.
template <int CIN, int THREADS = 256, int STRIDE = kPixStride>
struct Halo {
    static constexpr int kPerPixel = CIN / 8, kChunks = kHalo * kHalo * kPerPixel, kRegs = (kChunks + THREADS - 1) / THREADS;
    uint4 v[kRegs];
    __device__ __forceinline__ void load(const __bf16* __restrict__ in, int n, int H, int W, int y0, int x0) {
        const __bf16* img = in + size_t(n) * H * W * CIN;
#pragma unroll
        for (int k = 0; k < kRegs; k++) {
            const int c = threadIdx.x + k * THREADS, pix = c / kPerPixel, ch = c % kPerPixel;
            const int hy = pix / kHalo, hx = pix - hy * kHalo;
            const int gy = y0 + hy - 1, gx = x0 + hx - 1;
            v[k] = make_uint4(0u, 0u, 0u, 0u);
            if (c < kChunks && unsigned(gy) < unsigned(H) && unsigned(gx) < unsigned(W))
                v[k] = *reinterpret_cast<const uint4*>(img + (size_t(gy) * W + gx) * CIN + ch * 8);
        }
    }
    __device__ __forceinline__ void store(__bf16* tile) const {
#pragma unroll
        for (int k = 0; k < kRegs; k++) {
            const int c = threadIdx.x + k * THREADS;
            if (c < kChunks)
                *reinterpret_cast<uint4*>(tile + (c / kPerPixel) * STRIDE + (c % kPerPixel) * 8) = v[k];
        }
    }
    // zeroes the channels of the tile that store() leaves (once: they stay)
    static __device__ __forceinline__ void clearRest(__bf16* tile) {
        constexpr int kRest = kC / 8 - kPerPixel;
        if (kRest == 0) return;
        for (int i = threadIdx.x; i < kHalo * kHalo * kRest; i += THREADS)
            *reinterpret_cast<uint4*>(tile + i / max(kRest, 1) * STRIDE + CIN + i % max(kRest, 1) * 8) =
                make_uint4(0u, 0u, 0u, 0u);
    }
};

// The nine taps of a 3x3 convolution for one wave: output rows wave * 4 .. + 3 of the staged tile, acc[row][N tile].
// The MFMA takes the weights as its A operand and the pixels as B, so the 16x16 result is channels x pixels: lane
// (m, kb) holds output channels kb * 8 + nt * 4 + 0..3 of pixel m of the tile row (k_swizzleWeights orders the rows of
// its fragments so). FLIP mirrors the taps (the backward data pass).
//
// Bound by LDS reads: a 1-KB pixel operand feeds two MFMAs, and at 128 B per cycle the four waves' reads would take as
// long as their MFMAs. So each operand is read once and used by every output row it is a tap of (18 reads for 72
// MFMAs instead of 36), in an order that keeps every accumulator's taps ascending: results are those of a plain loop
// over the taps, bit for bit. FLIP is a template parameter because only then do the reads coincide at compile time.
template <bool FLIP>
__device__ __forceinline__ void convTaps(const __bf16* tile, const bf16x8 (&B)[9][2], int wave, int m, int kb,
                                         f32x4 (&acc)[4][2]) {
#pragma unroll
    for (int mt = 0; mt < 4; mt++) acc[mt][0] = acc[mt][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 6; r++) {
        const int hy = FLIP ? 5 - r : r;  // staged row of the wave's six
#pragma unroll
        for (int kx = 0; kx < 3; kx++) {
            const int hx = FLIP ? 2 - kx : kx;
            const bf16x8 A =
                *reinterpret_cast<const bf16x8*>(tile + ((wave * 4 + hy) * kHalo + (m + hx)) * kPixStride + kb * 8);
#pragma unroll
            for (int mt = 0; mt < 4; mt++) {
                const int ky = FLIP ? 2 - (hy - mt) : hy - mt;
                if (ky < 0 || ky > 2) continue;
                acc[mt][0] = mfma16(B[ky * 3 + kx][0], A, acc[mt][0]);
                acc[mt][1] = mfma16(B[ky * 3 + kx][1], A, acc[mt][1]);
            }
        }
    }
}

__device__ __forceinline__ void loadFragments(const bf16x8* __restrict__ wsw, int lane, bf16x8 (&B)[9][2]) {
#pragma unroll
    for (int t = 0; t < 9; t++) {
        B[t][0] = wsw[(t * 2 + 0) * 64 + lane];
        B[t][1] = wsw[(t * 2 + 1) * 64 + lane];
    }
}

__device__ __forceinline__ void loadBias(const float* __restrict__ bias, int kb, float (&bco)[2][4]) {
#pragma unroll
    for (int nt = 0; nt < 2; nt++)
#pragma unroll
        for (int i = 0; i < 4; i++) bco[nt][i] = bias[kb * 8 + nt * 4 + i];
}

// Stores the wave's four output rows from row y on, pixel column x, with the layer's epilogue (k_conv3x3): a lane's
// eight channels in one 16-byte store, so a wave writes whole lines (as two 8-byte stores per lane, each
// instruction half of every pixel, a hidden layer took 57 us at 1920x1080 instead of 55).
template <int EPI>
__device__ __forceinline__ void storeTile(const f32x4 (&acc)[4][2], const float (&bco)[2][4],
                                          const __bf16* __restrict__ mask, void* __restrict__ out, int n, int H, int W,
                                          int yw, int x, int kb, size_t outPixels) {
#pragma unroll
    for (int mt = 0; mt < 4; mt++) {
        const int y = yw + mt;
        if (y >= H || x >= W) continue;
        const size_t o = ((size_t(n) * H + y) * W + x) * kC + kb * 8;
        if (EPI == EPI_LINEAR_F32) {
            // a caller's buffer: of any float alignment, and of outPixels pixels
            if (o >= outPixels * kC) continue;
            float* dst = reinterpret_cast<float*>(out) + o;
#pragma unroll
            for (int i = 0; i < 8; i++) dst[i] = acc[mt][i >> 2][i & 3] + bco[i >> 2][i & 3];
        } else {
            bf16x8 r;
            if (EPI == EPI_RELU_BF16) {
#pragma unroll
                for (int i = 0; i < 8; i++) r[i] = (__bf16)fmaxf(acc[mt][i >> 2][i & 3] + bco[i >> 2][i & 3], 0.0f);
            } else {
                const bf16x8 mv = *reinterpret_cast<const bf16x8*>(mask + o);
#pragma unroll
                for (int i = 0; i < 8; i++) r[i] = (__bf16)((float)mv[i] > 0.0f ? acc[mt][i >> 2][i & 3] : 0.0f);
            }
            *reinterpret_cast<bf16x8*>(reinterpret_cast<__bf16*>(out) + o) = r;
        }
    }
}

// One 3x3 convolution layer over [N, H, W, 32] bf16 activations (persistent over 16x16 tiles).
//   EPI_RELU_BF16   out = bf16(max(conv + bias, 0))                      hidden layers
//   EPI_LINEAR_F32  out = f32(conv + bias)                               the logits
//   EPI_MASK_BF16   out = bf16(conv * (mask > 0))                        backward data pass through the layer below's
//                                                                        ReLU: mirrored taps, and the fragments hold
//                                                                        the transposed weights
// wsw: 9 taps x 2 N tiles x 64 lanes of bf16x8 fragments. CIN: channels per input pixel in memory (the rest are zero).
// Bound by memory: 128 B per pixel and layer, 1.4 times that with the halo. One hidden layer at 1920x1080: 99 us with
// each halo staged in turn and tiles dealt out in order, 85 us with each operand read once (convTaps), 69 us with the
// next halo prefetched and neighbouring tiles on one XCD, 55 us with 16-byte stores (storeTile) and two workgroups per
// CU (4.8 TB/s of compulsory bytes, what a large copy reaches here; 695 TFLOP/s).
template <int EPI, int CIN = kC>
__device__ __forceinline__ void convLayer(const __bf16* __restrict__ in, const bf16x8* __restrict__ wsw,
                                          const float* __restrict__ bias, const __bf16* __restrict__ mask,
                                          void* __restrict__ out, int N, int H, int W, size_t outPixels = 0) {
    __shared__ __attribute__((aligned(16))) __bf16 tile[kHalo * kHalo * kPixStride];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kb = lane >> 4;
    bf16x8 B[9][2];
    loadFragments(wsw, lane, B);
    float bco[2][4] = {};
    if (EPI != EPI_MASK_BF16) loadBias(bias, kb, bco);
    Halo<CIN>::clearRest(tile);
    TileWalk walk(N, H, W);
    Halo<CIN> halo;
    if (walk.valid()) halo.load(in, walk.n, H, W, walk.y0, walk.x0);
    while (walk.valid()) {
        const int n = walk.n, y0 = walk.y0, x0 = walk.x0;
        __syncthreads();  // the previous tile's LDS reads are done
        halo.store(tile);
        __syncthreads();
        walk.next();
        if (walk.valid()) halo.load(in, walk.n, H, W, walk.y0, walk.x0);
        f32x4 acc[4][2];
        convTaps<EPI == EPI_MASK_BF16>(tile, B, wave, m, kb, acc);
        storeTile<EPI>(acc, bco, mask, out, n, H, W, y0 + wave * 4, x0 + m, kb, outPixels);
    }
}

template <int EPI, int CIN>
__global__ __launch_bounds__(256) void k_conv3x3(const __bf16* __restrict__ in, const bf16x8* __restrict__ wsw,
                                                 const float* __restrict__ bias, const __bf16* __restrict__ mask,
                                                 void* __restrict__ out, int N, int H, int W) {
    convLayer<EPI, CIN>(in, wsw, bias, mask, out, N, H, W);
}

// Input features [N, 15, H, W] f32 -> bf16 network channels. Radiance (0-2) and radiance variance
// (11-13) enter as log(1 + max(v, 0)). The screen-space depth gradient (9-10) is A / sqrt(1 - A^2) of the averaged
// view-space normal component A (Clouds.glsl:296): +-inf where the normal lies on a view axis and NaN where rounding
// puts |A| above 1, so it is clamped to +-kGradientClamp. Any other non-finite input enters as 0: one NaN would
// otherwise spread through the 3x3 receptive fields of all six layers.
constexpr float kGradientClamp = 16.0f;

__device__ __forceinline__ __bf16 packFeature(int c, float x) {
    if (c == 9 || c == 10) {
        x = x != x ? 0.0f : fminf(fmaxf(x, -kGradientClamp), kGradientClamp);
    } else {
        if (!__builtin_isfinite(x)) x = 0.0f;
        if (c <= 2 || (c >= 11 && c <= 13)) x = log1pf(fmaxf(x, 0.0f));
    }
    return (__bf16)x;
}

// [N, H, W, 16] bf16 network inputs (channel 15 zero) of a pixel per thread; clears *loss (nullable) for the head, which
// runs behind this kernel. 32 B per pixel: the first layer's other 16 input channels are zeros it need not read.
// (Packing inside the first layer's staging took 135-150 us at 1920x1080 against 52 + 63 us: 18-pixel rows of 15 planes
// use little of each line, and the halo's logarithms are evaluated 1.3 times.)
__global__ void k_packFeatures(const float* __restrict__ f, __bf16* __restrict__ out, float* __restrict__ loss, int N,
                               int H, int W) {
    const size_t p = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t plane = size_t(H) * W;
    if (loss && p == 0) *loss = 0.0f;
    if (p >= size_t(N) * plane) return;
    const size_t n = p / plane, q = p - n * plane;
    bf16x8 v[2];
#pragma unroll
    for (int c = 0; c < kKpnPacked; c++)
        v[c >> 3][c & 7] = c < kKpnInputs ? packFeature(c, f[(n * kKpnInputs + c) * plane + q]) : (__bf16)0.0f;
#pragma unroll
    for (int k = 0; k < 2; k++) reinterpret_cast<bf16x8*>(out + p * kKpnPacked)[k] = v[k];
}

// What the last forward pass's final layer ran with, for the logits on demand: the image batch's shape, the layer's
// bias and its weight fragments (kept because the parameters may be updated before the logits are asked for).
struct KpnLastForward {
    int N, H, W, pad;
    float bias[kC];
    bf16x8 frag[9 * 2 * 64];
};
static_assert(sizeof(KpnLastForward) <= kKpnLastForwardBytes, "size of the last-forward record");

// Last layer and head: the 25 logits of every pixel stay in LDS, where the softmax and the 5x5 filter of the noisy
// radiance [N, 3, H, W] (zero outside the image) take them; pred [N, 3, H, W] (nullable) gets the filtered image. With
// a target (TRAIN): adds sum((pred - t)^2 / (t^2 + 0.01)) / (3 N H W) to *loss and writes the logits' gradient dZ
// [N, H, W, 32] bf16 (zero in the padding channels).
// Bound by the layer's own input; as kernels of their own, the layer and the head wrote and read 128 B of f32 logits a
// pixel (1920x1080: 90 + 90 us, now 74 us; 98 us before the noisy pixels were prefetched too).
constexpr int kLogitStride = 36;  // floats per pixel: 16-byte rows whose float4 reads hit different banks
constexpr int kNoisyTile = kTile + 4;

template <bool TRAIN>
__global__ __launch_bounds__(256, 2) void k_convHead(const __bf16* __restrict__ in, const bf16x8* __restrict__ wsw,
                                                  const float* __restrict__ bias, const float* __restrict__ noisy,
                                                  const float* __restrict__ target, float* __restrict__ pred,
                                                  __bf16* __restrict__ dz, float* __restrict__ loss,
                                                  KpnLastForward* __restrict__ last, int N, int H, int W) {
    // the staged input tile and the logits follow each other in the same LDS
    __shared__ __attribute__((aligned(16))) float lds[kTile * kTile * kLogitStride];
    static_assert(sizeof(lds) >= kHalo * kHalo * kPixStride * 2, "the input tile fits");
    __shared__ float noisyTile[3][kNoisyTile * kNoisyTile];
    __shared__ float red[4];
    __bf16* tile = reinterpret_cast<__bf16*>(lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, kb = lane >> 4;
    bf16x8 B[9][2];
    loadFragments(wsw, lane, B);
    float bco[2][4];
    loadBias(bias, kb, bco);
    if (blockIdx.x == 0 && wave == 0) {
#pragma unroll
        for (int t = 0; t < 18; t++) last->frag[t * 64 + lane] = B[t >> 1][t & 1];
        if (lane < kC) last->bias[lane] = bias[lane];
        if (lane == 0) {
            last->N = N;
            last->H = H;
            last->W = W;
        }
    }
    const size_t plane = size_t(H) * W;
    const float scale = 1.0f / (3.0f * float(size_t(N) * plane));
    float lossSum = 0.0f;
    float noisyNext[2][3];  // the next tile's noisy pixels, prefetched with its halo
    auto loadNoisy = [&](int n, int y0, int x0) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int i = tid + k * 256;
            const int gy = y0 + i / kNoisyTile - 2, gx = x0 + i % kNoisyTile - 2;
            const bool inside =
                i < kNoisyTile * kNoisyTile && unsigned(gy) < unsigned(H) && unsigned(gx) < unsigned(W);
#pragma unroll
            for (int c = 0; c < 3; c++)
                noisyNext[k][c] = inside ? noisy[(size_t(n) * 3 + c) * plane + size_t(gy) * W + gx] : 0.0f;
        }
    };
    TileWalk walk(N, H, W);
    Halo<kC> halo;
    if (walk.valid()) {
        halo.load(in, walk.n, H, W, walk.y0, walk.x0);
        loadNoisy(walk.n, walk.y0, walk.x0);
    }
    while (walk.valid()) {
        const int n = walk.n, y0 = walk.y0, x0 = walk.x0;
        __syncthreads();  // the previous tile's LDS reads are done
        halo.store(tile);
#pragma unroll
        for (int k = 0; k < 2; k++)
            if (tid + k * 256 < kNoisyTile * kNoisyTile)
#pragma unroll
                for (int c = 0; c < 3; c++) noisyTile[c][tid + k * 256] = noisyNext[k][c];
        __syncthreads();
        const int ty = tid / kTile, tx = tid % kTile, y = y0 + ty, x = x0 + tx;
        const size_t q = size_t(y) * W + x;
        float tgt[3] = {};
        if (TRAIN && y < H && x < W)
#pragma unroll
            for (int c = 0; c < 3; c++) tgt[c] = target[(size_t(n) * 3 + c) * plane + q];
        walk.next();
        if (walk.valid()) {
            halo.load(in, walk.n, H, W, walk.y0, walk.x0);
            loadNoisy(walk.n, walk.y0, walk.x0);
        }
        f32x4 acc[4][2];
        convTaps<false>(tile, B, wave, m, kb, acc);
        __syncthreads();  // the input tile has been read: the logits take its place
#pragma unroll
        for (int mt = 0; mt < 4; mt++)
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                const f32x4 v = acc[mt][nt];
                *reinterpret_cast<float4*>(lds + ((wave * 4 + mt) * kTile + m) * kLogitStride + kb * 8 + nt * 4) =
                    make_float4(v[0] + bco[nt][0], v[1] + bco[nt][1], v[2] + bco[nt][2], v[3] + bco[nt][3]);
            }
        __syncthreads();
        if (y >= H || x >= W) continue;
        float w[28];
#pragma unroll
        for (int k = 0; k < 7; k++)
            *reinterpret_cast<float4*>(w + k * 4) = *reinterpret_cast<const float4*>(lds + tid * kLogitStride + k * 4);
        float mx = -3.0e38f;
#pragma unroll
        for (int k = 0; k < kKpnTaps; k++) mx = fmaxf(mx, w[k]);
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < kKpnTaps; k++) {
            w[k] = __expf(w[k] - mx);
            s += w[k];
        }
        const float inv = 1.0f / s;
#pragma unroll
        for (int k = 0; k < kKpnTaps; k++) w[k] *= inv;
        float o[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < kKpnTaps; k++)
#pragma unroll
            for (int c = 0; c < 3; c++) o[c] += w[k] * noisyTile[c][(ty + k / 5) * kNoisyTile + tx + k % 5];
        if (pred)
#pragma unroll
            for (int c = 0; c < 3; c++) pred[(size_t(n) * 3 + c) * plane + q] = o[c];
        if (TRAIN) {
            float g[3];
            float lossPart = 0.0f;
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const float t = tgt[c];
                const float d = o[c] - t;
                const float den = 1.0f / (t * t + 0.01f);
                lossPart += d * d * den;
                g[c] = 2.0f * d * den * scale;
            }
            lossSum += lossPart * scale;
            float gw[kKpnTaps];
            float dot = 0.0f;
#pragma unroll
            for (int k = 0; k < kKpnTaps; k++) {
                const int e = (ty + k / 5) * kNoisyTile + tx + k % 5;
                gw[k] = g[0] * noisyTile[0][e] + g[1] * noisyTile[1][e] + g[2] * noisyTile[2][e];
                dot += w[k] * gw[k];
            }
            bf16x8 v[4];
#pragma unroll
            for (int k = 0; k < kC; k++) v[k >> 3][k & 7] = (__bf16)(k < kKpnTaps ? w[k] * (gw[k] - dot) : 0.0f);
            bf16x8* dst = reinterpret_cast<bf16x8*>(dz + (size_t(n) * plane + q) * kC);
#pragma unroll
            for (int k = 0; k < 4; k++) dst[k] = v[k];
        }
    }
    if (TRAIN) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) lossSum += __shfl_down(lossSum, off);
        if (lane == 0) red[wave] = lossSum;
        __syncthreads();
        if (tid == 0) atomicAdd(loss, (red[0] + red[1]) + (red[2] + red[3]));
    }
}

// The last forward pass's logits [N, H, W, 32] f32, from the final layer's input (the last of kKpnLayers activation
// buffers of N * H * W pixels each at `act`) and the weights it ran with, into a caller's buffer of outPixels pixels:
// what is beyond it is left out, pixels of it beyond the pass are 0.
__global__ __launch_bounds__(256) void k_convLogits(const __bf16* __restrict__ act,
                                                    const KpnLastForward* __restrict__ last, float* __restrict__ out,
                                                    size_t outPixels) {
    const int N = last->N, H = last->H, W = last->W;
    const size_t P = size_t(N) * H * W, first = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    for (size_t i = P * kC + first; i < outPixels * kC; i += size_t(gridDim.x) * blockDim.x) out[i] = 0.0f;
    if (P == 0) return;
    convLayer<EPI_LINEAR_F32>(act + size_t(kKpnLayers - 1) * P * kC, last->frag, last->bias, nullptr, out, N, H, W,
                              outPixels);
}

// Weight and bias gradients of one layer: dW[co][ci][tap] = sum over pixels p of dZ[p][co] * X[p + offset(tap)][ci] and
// db[co] = sum of dZ[p][co], a GEMM with a 9216-element output and the pixels as its reduction dimension, split over
// the workgroups (split-K). A workgroup of two waves stages per 16x16 tile the output gradient and the input halo as
// they lie in memory (channels innermost); the MFMA operands want eight consecutive pixels of one channel per lane,
// which the LDS transpose reads deliver (ds_read_b64_tr_b16: lane i of 16 gets column i of the 4x16 block whose row r
// lanes 4r..4r+3 address). Wave w takes input channels w * 16.. and all 32 output channels: 18 accumulators over all
// tiles the workgroup visits, and each input operand (two staged rows, one column shift) serves every tap and row pair
// it belongs to (67 operands for 144 MFMAs). The sums leave as the workgroup's row of partial sums:
// part[block][((tap * 4 + co / 16 * 2 + ci / 16) * 4 + i) * 64 + lane] (coalesced), then 32 bias sums;
// k_gradReduce adds the rows in a fixed order. (Splitting a tile's pixels over waves as well, with half as many rows,
// ran at the same speed, and Adam's division by |g| makes a different order of sums visible after a step.)
// Bound by LDS reads and, for the 1024 tiles of a 16 x 128 x 128 batch (two per workgroup), by the latency of the first
// tile. Measured there: 21.3 us + 5.1 us (bias) per layer with transposed copies of both operands built by 2-byte LDS
// writes, now 17.7 us for both.
constexpr int kWgradPartial = 9 * 4 * 4 * 64;          // weight sums of a workgroup's row (= 32 x 32 x 9)
constexpr int kWgradRow = kWgradPartial + kC;          // floats per row
constexpr int kWgradThreads = 128;
constexpr int kWgradStride = 48;                       // bf16 per staged pixel: 8 rows of a read hit different banks
static_assert(kWgradPartial == kKpnLayerParams, "one partial per weight");

typedef short s16x4 __attribute__((ext_vector_type(4)));

// Eight consecutive pixels of channel m (of the 16 from `p` on) for lane m: p = the first pixel's channels.
__device__ __forceinline__ bf16x8 transposed8(const __bf16* p, int m) {
    typedef __attribute__((address_space(3))) s16x4* Lds;
    const __bf16* q = p + (m >> 2) * kWgradStride + (m & 3) * 4;
    union {
        s16x4 half[2];
        bf16x8 all;
    } u;
    u.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)(q));
    u.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((Lds)(q + 4 * kWgradStride));
    return u.all;
}

// wRows / bRows: workgroups that sum weight tiles (b, b + wRows, ...) and bias pixels (64 at b * 64, then at
// (b + bRows) * 64, ...).
template <int CIN>
__global__ __launch_bounds__(kWgradThreads) void k_weightGrad(const __bf16* __restrict__ x,
                                                              const __bf16* __restrict__ dz, float* __restrict__ part,
                                                              int N, int H, int W, int wRows, int bRows) {
    __shared__ __attribute__((aligned(16))) __bf16 dzS[kTile * kTile * kWgradStride];
    __shared__ __attribute__((aligned(16))) __bf16 xs[kHalo * kHalo * kWgradStride];
    const int tid = threadIdx.x, lane = tid & 63, nt = tid >> 6;
    const int m = lane & 15, kb = lane >> 4;
    float* row = part + size_t(blockIdx.x) * kWgradRow;
    if (int(blockIdx.x) < wRows) {
        f32x4 acc[9][2];
#pragma unroll
        for (int t = 0; t < 9; t++) acc[t][0] = acc[t][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        typedef Halo<CIN, kWgradThreads, kWgradStride> XHalo;
        XHalo::clearRest(xs);
        XHalo halo;
        constexpr int kDzRegs = kTile * kTile * 4 / kWgradThreads;
        uint4 dzv[kDzRegs];
        const int tilesX = (W + kTile - 1) / kTile, tilesY = (H + kTile - 1) / kTile;
        const int numTiles = N * tilesX * tilesY;
        auto load = [&](int ti) {
            const int n = ti / (tilesX * tilesY), r = ti - n * tilesX * tilesY;
            const int y0 = (r / tilesX) * kTile, x0 = (r % tilesX) * kTile;
            halo.load(x, n, H, W, y0, x0);
#pragma unroll
            for (int k = 0; k < kDzRegs; k++) {
                const int c = tid + k * kWgradThreads, pix = c >> 2, ch = c & 3;
                const int gy = y0 + pix / kTile, gx = x0 + pix % kTile;
                dzv[k] = make_uint4(0u, 0u, 0u, 0u);
                if (gy < H && gx < W)
                    dzv[k] = *reinterpret_cast<const uint4*>(dz + ((size_t(n) * H + gy) * W + gx) * kC + ch * 8);
            }
        };
        load(blockIdx.x);  // wRows is at most the number of tiles
        for (int ti = blockIdx.x; ti < numTiles; ti += wRows) {
            __syncthreads();  // the previous tile's LDS reads are done
            halo.store(xs);
#pragma unroll
            for (int k = 0; k < kDzRegs; k++) {
                const int c = tid + k * kWgradThreads;
                *reinterpret_cast<uint4*>(dzS + (c >> 2) * kWgradStride + (c & 3) * 8) = dzv[k];
            }
            __syncthreads();
            if (ti + wRows < numTiles) load(ti + wRows);
            bf16x8 A[8][2];  // [row pair][co tile]
#pragma unroll
            for (int r = 0; r < 17; r++) {  // staged rows r and r + 1
                if (r % 2 == 0 && r < 16)
#pragma unroll
                    for (int mt = 0; mt < 2; mt++)
                        A[r / 2][mt] = transposed8(dzS + (r / 2 * 32 + kb * 8) * kWgradStride + mt * 16, m);
#pragma unroll
                for (int kx = 0; kx < 3; kx++) {
                    const int pix = (r + (kb >> 1)) * kHalo + (kb & 1) * 8 + kx;
                    const bf16x8 Bv = transposed8(xs + pix * kWgradStride + nt * 16, m);
#pragma unroll
                    for (int ky = 0; ky < 3; ky++) {
                        const int ks = (r - ky) / 2;  // row pair of the tile whose tap row ky is these rows
                        if ((r - ky) % 2 != 0 || r - ky < 0 || ks > 7) continue;
#pragma unroll
                        for (int mt = 0; mt < 2; mt++)
                            acc[ky * 3 + kx][mt] = mfma16(A[ks][mt], Bv, acc[ky * 3 + kx][mt]);
                    }
                }
            }
        }
#pragma unroll
        for (int t = 0; t < 9; t++)
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int i = 0; i < 4; i++) row[((t * 4 + mt * 2 + nt) * 4 + i) * 64 + lane] = acc[t][mt][i];
    }
    if (int(blockIdx.x) >= bRows) return;
    // bias row: thread (pixel slot, 8-channel group), two slots each; the slots are added in order
    float(*red)[kC + 1] = reinterpret_cast<float(*)[kC + 1]>(xs);
    const size_t P = size_t(N) * H * W;
    const int c8 = tid & 3;
    float s[2][8] = {};
    for (int h = 0; h < 2; h++)
        for (size_t p = size_t(blockIdx.x) * 64 + (tid >> 2) + 32 * h; p < P; p += size_t(bRows) * 64) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(dz + p * kC + c8 * 8);
#pragma unroll
            for (int j = 0; j < 8; j++) s[h][j] += (float)v[j];
        }
    __syncthreads();  // the last tile's LDS reads are done
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int j = 0; j < 8; j++) red[(tid >> 2) + 32 * h][c8 * 8 + j] = s[h][j];
    __syncthreads();
    if (tid < kC) {
        float t = 0.0f;
        for (int k = 0; k < 64; k++) t += red[k][tid];
        row[kWgradPartial + tid] = t;
    }
}

// Sums the rows of every layer's k_weightGrad in a fixed order into dW [layer][co][ci][tap] and db [layer][co]: layer
// blockIdx.y, workgroups 0..143 own 64 weight columns each, workgroup 144 the 32 bias columns; each thread sums every
// 4th (weights) or 8th (biases) row with 8 loads in flight, then LDS combines the row groups. One launch for all six
// layers: six of 8.7 us became one of 18 us (113 MB of rows, much of it from the Infinity Cache).
constexpr int kGradReduceBlocks = kWgradPartial / 64 + 1;

__global__ __launch_bounds__(256) void k_gradReduce(const float* __restrict__ part, int wRows, int bRows,
                                                    size_t layerStride, float* __restrict__ dW,
                                                    float* __restrict__ db) {
    __shared__ float red[256];
    const int tid = threadIdx.x, layer = blockIdx.y;
    const bool bias = blockIdx.x == kGradReduceBlocks - 1;
    const int cols = bias ? kC : 64, groups = 256 / cols;
    const int col = tid % cols, g = tid / cols, rows = bias ? bRows : wRows;
    const float* src = part + layer * layerStride + (bias ? kWgradPartial : blockIdx.x * 64) + col;
    float s8[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    int r = g;
    for (; r + 7 * groups < rows; r += 8 * groups) {
#pragma unroll
        for (int j = 0; j < 8; j++) s8[j] += src[size_t(r + j * groups) * kWgradRow];
    }
    for (; r < rows; r += groups) s8[0] += src[size_t(r) * kWgradRow];
    red[tid] = ((s8[0] + s8[1]) + (s8[2] + s8[3])) + ((s8[4] + s8[5]) + (s8[6] + s8[7]));
    __syncthreads();
    if (g != 0) return;
    float t = 0.0f;
    for (int k = 0; k < groups; k++) t += red[k * cols + col];
    if (bias) {
        db[layer * kC + col] = t;
        return;
    }
    // partial column e = ((tap * 4 + co tile * 2 + ci tile) * 4 + i) * 64 + lane -> (co, ci, tap)
    const int e = blockIdx.x * 64 + col;
    const int lane = e & 63, i = (e >> 6) & 3, pair = (e >> 8) & 3, tap = e >> 10;
    const int co = (pair >> 1) * 16 + (lane >> 4) * 4 + i, ci = (pair & 1) * 16 + (lane & 15);
    dW[size_t(layer) * kKpnLayerParams + (co * kC + ci) * 9 + tap] = t;
}

// Adam on the FP32 master parameters (bias-corrected, as torch.optim.Adam without weight decay).
__global__ void k_adam(float* __restrict__ param, const float* __restrict__ grad, float* __restrict__ m1,
                       float* __restrict__ m2, int n, float lr, float beta1, float beta2, float eps, float bc1,
                       float bc2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = grad[i];
    const float a = beta1 * m1[i] + (1.0f - beta1) * g;
    const float b = beta2 * m2[i] + (1.0f - beta2) * g * g;
    m1[i] = a;
    m2[i] = b;
    param[i] -= lr * (a / bc1) / (sqrtf(b / bc2) + eps);
}

// Master weights [layer][co][ci][tap] f32 -> per-lane MFMA fragments: forward B[k = ci][n = co] and, for the backward
// data pass, transposed B[k = co][n = ci]; [layer][tap][N tile][lane][8] bf16 each. Column n of N tile t is channel
// (n / 4) * 8 + t * 4 + n % 4, so that a lane's four results of both tiles are eight consecutive channels (storeTile).
__global__ void k_swizzleWeights(const float* __restrict__ w, bf16x8* __restrict__ fwd, bf16x8* __restrict__ bwd,
                                 int layers) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;  // (layer, tap, nt, lane)
    if (i >= layers * 9 * 2 * 64) return;
    const int lane = i & 63, nt = (i >> 6) & 1, t = (i >> 7) % 9, layer = i / (9 * 128);
    const float* wl = w + size_t(layer) * kKpnLayerParams;
    bf16x8 f, b;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int kk = (lane >> 4) * 8 + j, nn = ((lane & 15) >> 2) * 8 + nt * 4 + (lane & 3);
        f[j] = (__bf16)wl[(nn * kC + kk) * 9 + t];  // co = nn, ci = kk
        b[j] = (__bf16)wl[(kk * kC + nn) * 9 + t];  // co = kk, ci = nn
    }
    fwd[i] = f;
    bwd[i] = b;
}

__global__ void k_zeroF32(float* p, size_t n) {
    const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

static unsigned blocksFor(size_t n, int per = 256) { return unsigned((n + per - 1) / per); }

static unsigned tileBlocks(int N, int H, int W, int blocks) {
    const int tiles = N * ((H + kTile - 1) / kTile) * ((W + kTile - 1) / kTile);
    return unsigned(tiles < blocks ? tiles : blocks);
}

hipError_t launchKpnConv(bool first, const void* in, const void* wsw, const float* bias, void* out, int N, int H, int W,
                         int blocks, hipStream_t stream) {
    const dim3 grid(tileBlocks(N, H, W, blocks)), block(256);
    const __bf16* i = reinterpret_cast<const __bf16*>(in);
    const bf16x8* w = reinterpret_cast<const bf16x8*>(wsw);
    if (first)
        hipLaunchKernelGGL((k_conv3x3<EPI_RELU_BF16, kKpnPacked>), grid, block, 0, stream, i, w, bias, nullptr, out, N, H,
                           W);
    else
        hipLaunchKernelGGL((k_conv3x3<EPI_RELU_BF16, kC>), grid, block, 0, stream, i, w, bias, nullptr, out, N, H, W);
    return hipGetLastError();
}

hipError_t launchKpnConvBackward(const void* dz, const void* wsw, const void* mask, void* out, int N, int H, int W,
                                 int blocks, hipStream_t stream) {
    hipLaunchKernelGGL((k_conv3x3<EPI_MASK_BF16, kC>), dim3(tileBlocks(N, H, W, blocks)), dim3(256), 0, stream,
                       reinterpret_cast<const __bf16*>(dz), reinterpret_cast<const bf16x8*>(wsw), nullptr,
                       reinterpret_cast<const __bf16*>(mask), out, N, H, W);
    return hipGetLastError();
}

hipError_t launchKpnPack(const float* features, void* out, float* loss, int N, int H, int W, hipStream_t stream) {
    hipLaunchKernelGGL(k_packFeatures, dim3(blocksFor(size_t(N) * H * W)), dim3(256), 0, stream, features,
                       reinterpret_cast<__bf16*>(out), loss, N, H, W);
    return hipGetLastError();
}

hipError_t launchKpnConvHead(const void* in, const void* wsw, const float* bias, const float* noisy,
                             const float* target, float* pred, void* dz, float* loss, void* last, int N, int H, int W,
                             int blocks, hipStream_t stream) {
    const dim3 grid(tileBlocks(N, H, W, blocks)), block(256);
    const __bf16* i = reinterpret_cast<const __bf16*>(in);
    const bf16x8* w = reinterpret_cast<const bf16x8*>(wsw);
    __bf16* d = reinterpret_cast<__bf16*>(dz);
    KpnLastForward* l = reinterpret_cast<KpnLastForward*>(last);
    if (target)
        hipLaunchKernelGGL(k_convHead<true>, grid, block, 0, stream, i, w, bias, noisy, target, pred, d, loss, l, N, H,
                           W);
    else
        hipLaunchKernelGGL(k_convHead<false>, grid, block, 0, stream, i, w, bias, noisy, target, pred, d, loss, l, N, H,
                           W);
    return hipGetLastError();
}

hipError_t launchKpnLogits(const void* act, const void* last, float* out, size_t outPixels, int blocks,
                           hipStream_t stream) {
    hipLaunchKernelGGL(k_convLogits, dim3(unsigned(blocks)), dim3(256), 0, stream,
                       reinterpret_cast<const __bf16*>(act), reinterpret_cast<const KpnLastForward*>(last), out,
                       outPixels);
    return hipGetLastError();
}

size_t kpnGradWorkFloats(int blocks) { return size_t(blocks) * kWgradRow * kKpnLayers; }

// Rows of weight sums (workgroups with tiles) and of bias sums (workgroups with 64 pixels) of `blocks` at most.
static int weightRows(int N, int H, int W, int blocks) { return int(tileBlocks(N, H, W, blocks)); }
static int biasRows(int N, int H, int W, int blocks) {
    const size_t b = (size_t(N) * H * W + 63) / 64;
    return int(b < size_t(blocks) ? b : size_t(blocks));
}

hipError_t launchKpnWeightGrad(int layer, const void* x, const void* dz, int N, int H, int W, int blocks, float* work,
                               hipStream_t stream) {
    const int wRows = weightRows(N, H, W, blocks), bRows = biasRows(N, H, W, blocks);
    const dim3 grid(unsigned(wRows > bRows ? wRows : bRows)), block(kWgradThreads);
    const __bf16* in = reinterpret_cast<const __bf16*>(x);
    const __bf16* d = reinterpret_cast<const __bf16*>(dz);
    float* part = work + size_t(layer) * blocks * kWgradRow;
    if (layer == 0)
        hipLaunchKernelGGL(k_weightGrad<kKpnPacked>, grid, block, 0, stream, in, d, part, N, H, W, wRows, bRows);
    else
        hipLaunchKernelGGL(k_weightGrad<kC>, grid, block, 0, stream, in, d, part, N, H, W, wRows, bRows);
    return hipGetLastError();
}

hipError_t launchKpnGradReduce(const float* work, int N, int H, int W, int blocks, float* dW, float* db,
                               hipStream_t stream) {
    hipLaunchKernelGGL(k_gradReduce, dim3(kGradReduceBlocks, kKpnLayers), dim3(256), 0, stream, work,
                       weightRows(N, H, W, blocks), biasRows(N, H, W, blocks), size_t(blocks) * kWgradRow, dW, db);
    return hipGetLastError();
}

hipError_t launchKpnAdam(float* param, const float* grad, float* m1, float* m2, int n, float lr, float beta1,
                         float beta2, float eps, float bc1, float bc2, hipStream_t stream) {
    hipLaunchKernelGGL(k_adam, dim3(blocksFor(size_t(n))), dim3(256), 0, stream, param, grad, m1, m2, n, lr, beta1,
                       beta2, eps, bc1, bc2);
    return hipGetLastError();
}

hipError_t launchKpnSwizzle(const float* w, void* fwd, void* bwd, int layers, hipStream_t stream) {
    hipLaunchKernelGGL(k_swizzleWeights, dim3(blocksFor(size_t(layers) * 9 * 128)), dim3(256), 0, stream, w,
                       reinterpret_cast<bf16x8*>(fwd), reinterpret_cast<bf16x8*>(bwd), layers);
    return hipGetLastError();
}

hipError_t launchKpnZero(float* p, size_t n, hipStream_t stream) {
    hipLaunchKernelGGL(k_zeroF32, dim3(blocksFor(n)), dim3(256), 0, stream, p, n);
    return hipGetLastError();
}

}  // namespace crvpt
