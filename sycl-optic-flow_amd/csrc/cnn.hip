// cnn.hip -- the learned warm start of TV-L1 (no reference counterpart).
//
// A small fully convolutional network predicts the flow at the coarsest
// pyramid scale from that scale's I0, I1, Ix, Iy and It; the solver then
// starts from it instead of zero (the reference starts from zero,
// src/tvl1/sequential/tvl1.cpp:157-158).  Layers: conv3x3 5->C + ReLU,
// `hidden` x (conv3x3 C->C + ReLU), conv3x3 C->2; zero padding.
//
// Every convolution is an implicit GEMM on the bf16 MFMA
// (v_mfma_f32_16x16x32_bf16, fp32 accumulation), with M = pixels:
//   forward        Y[m][n]  = sum_(t,c) X[m + s(t)][c] W[n][t][c]
//   data gradient  dX[m][c] = sum_(t,n) dY[m - s(t)][n] W[n][t][c]
//   weight grad.   dW[n][t][c] = sum_m dY[m][n] X[m + s(t)][c]
// with tap offsets s(t) = (t/3 - 1, t%3 - 1).  Activations are NHWC fp32 in
// memory and rounded to bf16 (nearest even) as they enter an MFMA operand;
// the master weights are fp32 (Adam) with bf16 copies packed for the two
// GEMM orientations.  Every reduction runs in a fixed order, so a training
// run is deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <new>
#include <random>
#include <vector>

#include "amdflow.h"
#include "amdflow_debug.h"
#include "common.hpp"

namespace amdflow {
namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ __forceinline__ short to_bf16(float f)
{
    unsigned u;
    std::memcpy(&u, &f, 4);
    if ((u & 0x7F800000u) == 0x7F800000u) return (short)(u >> 16);   // inf / nan: truncate
    u += 0x7FFFu + ((u >> 16) & 1u);                                   // nearest even
    return (short)(u >> 16);
}

// gfx950 16x16x32 MFMA: lane l supplies row (l % 16) of A and column
// (l % 16) of B for k = 8*(l/16) .. +7, and receives column (l % 16), rows
// 4*(l/16) .. +3 of the 16x16 product (of_dbg_cnn_mfma checks this through
// k_conv_lds).
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// fp32 -> bf16, round to nearest even (v_cvt_pk_bf16_f32 on gfx950).
__device__ __forceinline__ bf16x8 to_bf16x8(f32x8 v) { return __builtin_convertvector(v, bf16x8); }

// GEMM-k layout of the packed weights: tap t, channel c at k = t*C + c, zero
// from 9*C on, the whole padded to a multiple of 32.
__host__ __device__ constexpr int pad_k(int c) { return (9 * c + 31) / 32 * 32; }

// Eight consecutive channels c8 .. c8+7 (zero past CX) of an NHWC pixel.
template <int CX>
__device__ __forceinline__ f32x8 load_channels(const float* __restrict__ X, long long pix, int c8)
{
    f32x8 v;
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = 0.0f;
    if constexpr (CX % 8 == 0) {
        const float4* q = reinterpret_cast<const float4*>(X + pix * CX + c8);
        const float4 v0 = q[0], v1 = q[1];
        v[0] = v0.x; v[1] = v0.y; v[2] = v0.z; v[3] = v0.w;
        v[4] = v1.x; v[5] = v1.y; v[6] = v1.z; v[7] = v1.w;
    } else {
        static_assert(CX <= 8, "one group of 8 channels");
#pragma unroll
        for (int j = 0; j < CX; j++) v[j] = X[pix * CX + j];
    }
    return v;
}

// Implicit-GEMM 3x3 convolution on the MFMA, 16-wide output tiles of NT*16
// channels.  A block (4 waves) computes a tile of 16 x TR pixels of one
// image, each wave TR/4 rows of 16 pixels (one MFMA row block each), from a
// (16+2) x (TR+2) bf16 input patch and the bf16 weights, both staged in LDS
// once.  Epilogue: + bias, ReLU, and/or zero where mask[m][n] <= 0 (the ReLU
// derivative of the layer below).
//
// Bound by the fp32 activations (each read once plus the halo, written
// once; 32 images of 68x120x32: 67 MB, 17.9 us, 3.7 TB/s) and at small
// batches by the latency of one tile, so every load of a tile is issued before
// the first is used: with branches around the loads they had gone out one by
// one (26.7 us; one image 9 us, now 3.8).  LDS rows are padded by 16 B so that
// 8 lanes' 16-byte reads fall on distinct banks.
//
// The 8 consecutive k of an MFMA lane are channels of one tap where CX is a
// multiple of 8: one 16-byte LDS read.  The 5- and 2-channel layers read them
// one by one, by a table of offsets (16 images of 68x120: the whole forward 82.1
// us, 84.4 with the offsets computed per lane): padding a tap to 8 channels instead would group the fp32 sums
// differently and, past 9*CX, multiply zero weights with pixels, which an
// infinite one turns into NaN.
template <int CX, int NT, int TR>
__global__ __launch_bounds__(256) void k_conv_lds(const float* __restrict__ X, int B, int H, int W,
                                                  const short* __restrict__ Wp, int N,
                                                  const float* __restrict__ bias, int sgn, int relu,
                                                  const float* __restrict__ mask,
                                                  float* __restrict__ Y)
{
    constexpr int CP = (CX + 7) / 8 * 8, KP = pad_k(CX), MB = TR / 4;
    constexpr bool kWhole = CX % 8 == 0;   // a lane's 8 k lie in one tap
    // shorts per pixel: rows of whole 16 bytes, or the channels and a zero in an
    // odd number of dwords (5 channels) or two (2 channels)
    constexpr int PW = 18, PP = PW * (TR + 2), PS = kWhole ? CP + 8 : CX / 2 * 2 + 2, WS = KP + 8;
    __shared__ __align__(16) short patch[PP * PS];
    __shared__ __align__(16) short wts[NT * 16 * WS];
    __shared__ __align__(16) short koff[kWhole ? 8 : KP];   // patch offset of every k
    const int tiles_x = (W + 15) / 16, tiles_y = (H + TR - 1) / TR;
    const int tile = blockIdx.x;
    const int b = tile / (tiles_x * tiles_y);
    const int r = tile - b * tiles_x * tiles_y;
    const int y0 = (r / tiles_x) * TR, x0 = (r % tiles_x) * 16;
    // input patch rows y0-1 .. y0+TR, columns x0-1 .. x0+16, zero outside; all
    // of a thread's loads are issued before its first LDS write
    constexpr int ITEMS = PP * (CP / 8), NI = (ITEMS + 255) / 256;
    // (positions outside read pixel 0 instead of branching around the load)
    f32x8 v[NI];
    bool in[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int e = (int)threadIdx.x + 256 * i;
        const int pix = e / (CP / 8), c8 = (e - pix * (CP / 8)) * 8;
        const int yy = y0 - 1 + pix / PW, xx = x0 - 1 + pix % PW;
        in[i] = e < ITEMS && yy >= 0 && yy < H && xx >= 0 && xx < W;
        v[i] = load_channels<CX>(X, in[i] ? ((long long)b * H + yy) * W + xx : 0, c8);
    }
    for (int e = threadIdx.x; e < NT * 16 * (KP / 8); e += 256) {
        const int n = e / (KP / 8), k8 = e - n * (KP / 8);
        *reinterpret_cast<s16x8*>(wts + n * WS + 8 * k8) = reinterpret_cast<const s16x8*>(Wp)[e];
    }
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int e = (int)threadIdx.x + 256 * i;
        const int pix = e / (CP / 8), c8 = (e - pix * (CP / 8)) * 8;
        const bf16x8 q = in[i] ? to_bf16x8(v[i]) : bf16x8{};
        if (e >= ITEMS) continue;
        if constexpr (kWhole) *reinterpret_cast<bf16x8*>(patch + pix * PS + c8) = q;
        else {
            const s16x8 w = __builtin_bit_cast(s16x8, q);
#pragma unroll
            for (int d = 0; d < PS; d += 2) *reinterpret_cast<s16x2*>(patch + pix * PS + d) = s16x2{w[d], w[d + 1]};
        }
    }
    if constexpr (!kWhole) {   // past the last tap the zero behind the channels
        static_assert(KP <= 256, "one entry per thread");
        const int k = threadIdx.x, tap = k / CX, c = k - tap * CX;
        if (k < KP) koff[k] = k < 9 * CX ? sgn * ((tap / 3 - 1) * PW + (tap % 3 - 1)) * PS + c : CX;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 15, kg = lane >> 4;
    f32x4 acc[MB][NT];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    const short* pbase = patch + ((wave * MB + 1) * PW + row + 1) * PS;
#pragma unroll
    for (int k0 = 0; k0 < KP; k0 += 32) {
        const int k = k0 + 8 * kg;
        // (the 16-channel layer of the test entry point has k past its taps)
        const int tap = CX % 32 == 0 ? k0 / CX : k / CX, c = CX % 32 == 0 ? k0 % CX + 8 * kg : k % CX;
        const int off = kWhole && k < 9 * CX ? sgn * ((tap / 3 - 1) * PW + (tap % 3 - 1)) * PS + c : 0;
        s16x8 offs{};
        if constexpr (!kWhole) offs = *reinterpret_cast<const s16x8*>(koff + k);
        bf16x8 w[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) w[t] = *reinterpret_cast<const bf16x8*>(wts + (t * 16 + row) * WS + k);
#pragma unroll
        for (int m = 0; m < MB; m++) {
            const short* p = pbase + m * PW * PS;
            bf16x8 a;
            if constexpr (kWhole) {
                a = *reinterpret_cast<const bf16x8*>(p + off);
                if (9 * CX % 32 != 0 && k >= 9 * CX) a = bf16x8{};
            } else {
                s16x8 v8;
#pragma unroll
                for (int j = 0; j < 8; j++) v8[j] = p[offs[j]];
                a = __builtin_bit_cast(bf16x8, v8);
            }
#pragma unroll
            for (int t = 0; t < NT; t++) acc[m][t] = mfma32(a, w[t], acc[m][t]);
        }
    }
    // accumulator: column n = t*16 + row, rows (pixels) x0 + 4*kg + j of image row
    if (relu || bias) {
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const float bn = bias && t * 16 + row < N ? bias[t * 16 + row] : 0.0f;
#pragma unroll
            for (int m = 0; m < MB; m++)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float q = acc[m][t][j] + bn;
                    acc[m][t][j] = relu && !(q > 0.0f) ? 0.0f : q;
                }
        }
    }
#pragma unroll
    for (int m = 0; m < MB; m++) {
        const int yy = y0 + wave * MB + m;
        if (yy >= H) break;
        const long long o0 = (((long long)b * H + yy) * W + x0 + 4 * kg) * N + row;
        bool ok[4][NT];
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int t = 0; t < NT; t++) ok[j][t] = x0 + 4 * kg + j < W && t * 16 + row < N;
        if (mask) {
            float mk[4][NT];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int t = 0; t < NT; t++) mk[j][t] = mask[ok[j][t] ? o0 + j * N + t * 16 : 0];
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int t = 0; t < NT; t++)
                    if (!(mk[j][t] > 0.0f)) acc[m][t][j] = 0.0f;
        }
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int t = 0; t < NT; t++)
                if (ok[j][t]) Y[o0 + j * N + t * 16] = acc[m][t][j];
    }
}

// Weight- and bias-gradient partials of one layer.  dW[n][t][c] is a GEMM over
// pixels: a block walks tiles of 8 x 16 pixels (blockIdx.x, + gridDim.x, ..)
// and keeps its whole dW in MFMA accumulators, the NT*16 x 16 column tiles
// dealt to its 4 waves.  Per tile dY^T and X^T are staged in LDS as bf16 with
// 8 consecutive pixels of a channel per 16 bytes, which is what one lane of
// an MFMA operand holds; X^T three times, shifted by the taps' dx, so that
// every tap reads aligned.  part: [blocks][NT*16][Kpad] with k = t*CX + c.
// The bias gradient is the fp32 sum of dY, taken on the way to LDS.
// Positions of a tile outside the image have dY = 0 and X = 0: a pixel inside
// that such a position's taps would reach must not count even where it is
// infinite (0 * inf is NaN), so the operand that such a position multiplies is
// zero by the position of dY, not of X.
//
// Bound by reading dY and X once (fp32; 67 MB per 32->32 layer at 32 x 68 x
// 120 pixels).  The earlier kernel formed one 16x16
// tile per block and so read both once per column tile: 139 us per 32->32
// layer of 32 x 68 x 120 pixels, and 122 us for the bias sums.
constexpr int kWgRows = 16;          // tile height in pixels
constexpr int kWgMaxBlocks = 768;    // three per CU; bounds the partials

template <int CX, int N>
__global__ __launch_bounds__(256) void k_wgrad(const float* __restrict__ dY,
                                               const float* __restrict__ X, int B, int H, int W,
                                               int ntiles, int Kpad, float* __restrict__ part,
                                               float* __restrict__ bpart)
{
    constexpr int NT = (N + 15) / 16;
    constexpr int T = kWgRows, XR = T + 2, YR = T + 1;   // YR: one row of padding against bank conflicts
    constexpr int COLS = (9 * CX + 15) / 16, CW = (COLS + 3) / 4;
    __shared__ __align__(16) short xs[3][CX][XR][8];
    __shared__ __align__(16) short ys[NT * 16][YR][8];
    __shared__ float sb[256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane & 15, kg = lane >> 4;
    const int tiles_x = (W + 7) / 8, tiles_y = (H + T - 1) / T;
    // LDS offset of this lane's column of each of the wave's column tiles, and
    // that for the first row past the image, whose upper taps reach the last
    // row inside: they read the row of zeros after it
    int xoff[CW], xbelow[CW];
#pragma unroll
    for (int i = 0; i < CW; i++) {
        const int k = min((wave + 4 * i) * 16 + row, 9 * CX - 1);   // past the end: computed, not read back
        const int t = k / CX, c = k - t * CX;
        xoff[i] = ((t % 3) * CX + c) * XR * 8 + (t / 3) * 8;
        xbelow[i] = xoff[i] + (t / 3 == 0 ? 8 : 0);
    }
    f32x4 acc[CW][NT];
#pragma unroll
    for (int i = 0; i < CW; i++)
#pragma unroll
        for (int t = 0; t < NT; t++) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    // rows past N stay zero
    for (int e = threadIdx.x; e < NT * 16 * YR; e += 256)
        *reinterpret_cast<bf16x8*>(&ys[0][0][0] + 8 * e) = bf16x8{};
    float bsum = 0.0f;
    const int yn = (int)threadIdx.x % N;   // 256 % N == 0: a thread's dY items share the channel
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int b = tile / (tiles_x * tiles_y);
        const int r = tile - b * tiles_x * tiles_y;
        const int y0 = (r / tiles_x) * T, x0 = (r % tiles_x) * 8;
        // positions outside the image load a pixel inside instead of branching
        // around the load, and are zeroed afterwards
        const bool xedge = x0 == 0 || x0 + 9 > W;   // uniform
        constexpr int XI = (XR * CX + 255) / 256;
        float xv[XI][10];
        bool xin[XI];
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int e = (int)threadIdx.x + 256 * i;
            const int pr = e / CX, c = e - pr * CX;
            const int yy = y0 - 1 + pr;
            xin[i] = e < XR * CX && yy >= 0 && yy < H;
            const float* p = X + (xin[i] ? ((long long)b * H + yy) * W * CX : 0) + c;
#pragma unroll
            for (int j = 0; j < 10; j++) xv[i][j] = p[min(max(x0 - 1 + j, 0), W - 1) * CX];
            if (xedge) {
#pragma unroll
                for (int j = 0; j < 10; j++)
                    if (x0 - 1 + j < 0 || x0 - 1 + j >= W) xv[i][j] = 0.0f;
            }
        }
        constexpr int YI = (T * N + 255) / 256;
        float yv[YI][8];
        bool yin[YI];
#pragma unroll
        for (int i = 0; i < YI; i++) {
            const int e = (int)threadIdx.x + 256 * i, yy = y0 + e / N;
            yin[i] = e < T * N && yy < H;
            const float* p = dY + (yin[i] ? ((long long)b * H + yy) * W * N : 0) + yn;
#pragma unroll
            for (int j = 0; j < 8; j++) yv[i][j] = p[min(x0 + j, W - 1) * N];
            if (xedge) {
#pragma unroll
                for (int j = 0; j < 8; j++)
                    if (x0 + j >= W) yv[i][j] = 0.0f;
            }
        }
        __syncthreads();   // the previous tile's operands have been read
#pragma unroll
        for (int i = 0; i < XI; i++) {
            const int e = (int)threadIdx.x + 256 * i;
            const int pr = e / CX, c = e - pr * CX;
            if (e < XR * CX) {
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    f32x8 v;
#pragma unroll
                    for (int j = 0; j < 8; j++) v[j] = xv[i][d + j];
                    // dY past the last column: X there is zero by now but for
                    // its left taps
                    if (d == 0 && x0 + 8 > W) {   // uniform
#pragma unroll
                        for (int j = 1; j < 8; j++) v[j] = x0 + j < W ? v[j] : 0.0f;
                    }
                    *reinterpret_cast<bf16x8*>(&xs[d][c][pr][0]) = xin[i] ? to_bf16x8(v) : bf16x8{};
                }
            }
        }
#pragma unroll
        for (int i = 0; i < YI; i++) {
            const int e = (int)threadIdx.x + 256 * i;
            f32x8 v;
            float s = 0.0f;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                v[j] = yin[i] ? yv[i][j] : 0.0f;
                s += v[j];
            }
            bsum += s;
            if (e < T * N) *reinterpret_cast<bf16x8*>(&ys[yn][e / N][0]) = to_bf16x8(v);
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < T / 4; ks++) {   // 32 pixels: 4 rows of 8
            const int pr = ks * 4 + kg;
            const bool below = pr == H - y0;   // the first row past the image
            bf16x8 a[NT];
#pragma unroll
            for (int t = 0; t < NT; t++) a[t] = *reinterpret_cast<const bf16x8*>(&ys[t * 16 + row][pr][0]);
#pragma unroll
            for (int i = 0; i < CW; i++) {
                if (wave + 4 * i >= COLS) break;   // wave-uniform
                const int off = below ? xbelow[i] : xoff[i];
                const bf16x8 x = *reinterpret_cast<const bf16x8*>(&xs[0][0][0][0] + off + pr * 8);
#pragma unroll
                for (int t = 0; t < NT; t++) acc[i][t] = mfma32(a[t], x, acc[i][t]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < CW; i++) {
        const int col = wave + 4 * i;
        if (col >= COLS) break;
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int j = 0; j < 4; j++)
                part[((size_t)blockIdx.x * (NT * 16) + t * 16 + 4 * kg + j) * Kpad + col * 16 + row] = acc[i][t][j];
    }
    sb[threadIdx.x] = bsum;
    __syncthreads();
    if ((int)threadIdx.x < N) {
        float s = sb[threadIdx.x];
        for (int q = (int)threadIdx.x + N; q < 256; q += N) s += sb[q];
        bpart[(size_t)blockIdx.x * N + threadIdx.x] = s;
    }
}

// dW and db: sums of the partials in a fixed order.  A block sums 64 outputs,
// 16 interleaved groups of partials each, then the groups in order (a single
// thread per output took 16 us per layer, one chain of 256 loads).
__global__ __launch_bounds__(1024) void k_grad_reduce(const float* __restrict__ part, int parts, int Npad,
                                                      int Kpad, int N, int K, float* __restrict__ dW,
                                                      const float* __restrict__ bpart,
                                                      float* __restrict__ db)
{
    __shared__ float sh[16][64];
    const int o = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int idx = blockIdx.x * 64 + o;
    float s = 0.0f;
    if (idx < N * K) {
        const int n = idx / K, k = idx - n * K;
        const float* p = part + (size_t)n * Kpad + k;
#pragma unroll 8
        for (int sp = q; sp < parts; sp += 16) s += p[(size_t)sp * Npad * Kpad];
    } else if (idx < N * K + N) {
#pragma unroll 8
        for (int sp = q; sp < parts; sp += 16) s += bpart[(size_t)sp * N + (idx - N * K)];
    }
    sh[q][o] = s;
    __syncthreads();
    if (q == 0 && idx < N * K + N) {
#pragma unroll
        for (int g = 1; g < 16; g++) s += sh[g][o];
        if (idx < N * K) dW[idx] = s;
        else db[idx - N * K] = s;
    }
}

// Mean-squared flow error against planar targets T[b][2][H*W]:
// L = sum (Y - T)^2 / (2 M), dY = (Y - T) / M (M pixels); per-block double
// partial sums of the squared error.
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ Y, const float* __restrict__ T,
                                             long long M, int HW, float invM, float* __restrict__ dY,
                                             double* __restrict__ part)
{
    __shared__ double sh[256];
    double s = 0.0;
    for (long long i = blockIdx.x * 256ll + threadIdx.x; i < 2 * M; i += (long long)gridDim.x * 256) {
        const long long m = i >> 1;
        const int c = (int)(i & 1);
        const long long b = m / HW;
        const long long r = m - b * HW;
        const float d = Y[i] - T[(b * 2 + c) * HW + r];
        dY[i] = d * invM;
        s += (double)d * (double)d;
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// Sum of the block partials, one workgroup, fixed order (one thread took 51 us
// for 1024 of them, a chain of dependent loads).
__global__ __launch_bounds__(256) void k_sum_f64(const double* __restrict__ part, int n, double scale,
                                                 double* __restrict__ out)
{
    __shared__ double sh[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += part[i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sh[0] * scale;
}

// Adam (Kingma & Ba 2015) with bias-correction factors c1 = 1 - b1^t,
// c2 = 1 - b2^t.
__global__ __launch_bounds__(256) void k_adam(float* __restrict__ w, const float* __restrict__ g,
                                              float* __restrict__ m, float* __restrict__ v, int n,
                                              float lr, float b1, float b2, float eps, float c1,
                                              float c2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// bf16 packs of one layer's weights Wm[n][t][c] (N outputs, C inputs), zero
// in the padding:
//   fwd [Npad][pad_k(C)]: row n, k = t*C + c
//   bwd [Cpad][pad_k(N)]: row c, k = t*N + n
__global__ __launch_bounds__(256) void k_pack(const float* __restrict__ Wm, int N, int C, int Npad,
                                              int Cpad, short* __restrict__ fwd,
                                              short* __restrict__ bwd)
{
    const int Kf = pad_k(C), Kb = pad_k(N);
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < Npad * Kf) {
        const int n = idx / Kf, k = idx - n * Kf;
        fwd[idx] = (n < N && k < 9 * C) ? to_bf16(Wm[n * 9 * C + k]) : (short)0;
    }
    if (idx < Cpad * Kb) {
        const int c = idx / Kb, k = idx - c * Kb;
        const int t = k / N, n = k - t * N;
        bwd[idx] = (c < C && t < 9) ? to_bf16(Wm[(n * 9 + t) * C + c]) : (short)0;
    }
}

// Network input: I0, I1, Ix, Iy, It of one scale, /255.  Ix, Iy are
// centred differences of I1 (x0.5, clamped neighbours at the border).
__global__ __launch_bounds__(256) void k_features(const float* __restrict__ I0,
                                                  const float* __restrict__ I1, int H, int W,
                                                  float* __restrict__ X)
{
    const int idx = blockIdx.x * 256 + threadIdx.x;
    if (idx >= H * W) return;
    const int y = idx / W, x = idx - y * W;
    const int xl = x > 0 ? x - 1 : 0, xr = x < W - 1 ? x + 1 : W - 1;
    const int yu = y > 0 ? y - 1 : 0, yd = y < H - 1 ? y + 1 : H - 1;
    const float s = 1.0f / 255.0f;
    const float a = I0[idx], b = I1[idx];
    float* o = X + (size_t)idx * 5;
    o[0] = a * s;
    o[1] = b * s;
    o[2] = 0.5f * (I1[y * W + xr] - I1[y * W + xl]) * s;
    o[3] = 0.5f * (I1[yd * W + x] - I1[yu * W + x]) * s;
    o[4] = (b - a) * s;
}

// NHWC two-channel output -> planar [u1 | u2].
__global__ __launch_bounds__(256) void k_to_planar(const float* __restrict__ Y, int HW,
                                                   float* __restrict__ U)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= HW) return;
    U[i] = Y[2 * (size_t)i];
    U[HW + i] = Y[2 * (size_t)i + 1];
}

inline int pad16(int v) { return (v + 15) / 16 * 16; }
// From two 16x8-pixel tiles per CU on, the convolution takes them; below, 16x4
// tiles, whose workgroups are shorter and twice as many.  Measured per 32->32
// layer of 68x120 pixels (us, 16x8 / 16x4): batch 1 4.4 / 3.8, 4 5.3 / 5.1,
// 8 6.8 / 6.9, 16 10.5 / 10.9, 32 17.9 / 18.2 (16x16 tiles 10.2 and 19.1 at
// 16 and 32).
constexpr long long kConvTallTiles = 512;

inline int pad32(int v) { return (v + 31) / 32 * 32; }
inline unsigned blocks256(long long n)
{
    const long long g = (n + 255) / 256;
    return (unsigned)std::max<long long>(1, std::min<long long>(g, 1 << 20));
}

#define CNN_CHECK(name)                                     \
    do {                                                    \
        hipError_t e_ = hipGetLastError();                  \
        if (e_ != hipSuccess) {                             \
            record_hip_error(e_, name, __FILE__, __LINE__); \
            return OF_ERR_HIP;                              \
        }                                                   \
    } while (0)

template <int CX, int NT, int TR>
int launch_conv_tile(const float* X, int B, int H, int W, const short* Wp, int N, const float* bias, int sgn,
                     int relu, const float* mask, float* Y, hipStream_t st)
{
    const unsigned tiles = (unsigned)B * ((H + TR - 1) / TR) * ((W + 15) / 16);
    hipLaunchKernelGGL((k_conv_lds<CX, NT, TR>), dim3(tiles), dim3(256), 0, st, X, B, H, W, Wp, N, bias, sgn,
                       relu, mask, Y);
    CNN_CHECK("k_conv_lds");
    return OF_OK;
}

// Dispatch over the instantiated (input channels, output tiles) pairs and the
// tile height.
int launch_conv(const float* X, int B, int H, int W, int CX, const short* Wp, int N, const float* bias,
                int sgn, int relu, const float* mask, float* Y, hipStream_t st)
{
    const int NT = N <= 16 ? 1 : 2;
    if (N > 32) return OF_ERR_UNSUPPORTED;
    const bool tall = (long long)B * ((H + 7) / 8) * ((W + 15) / 16) >= kConvTallTiles;
#define CONV_CASE(cx, nt)                                                                            \
    if (CX == cx && NT == nt)                                                                        \
        return tall ? launch_conv_tile<cx, nt, 8>(X, B, H, W, Wp, N, bias, sgn, relu, mask, Y, st)  \
                    : launch_conv_tile<cx, nt, 4>(X, B, H, W, Wp, N, bias, sgn, relu, mask, Y, st);
    CONV_CASE(5, 2)
    CONV_CASE(32, 2)
    CONV_CASE(32, 1)
    CONV_CASE(2, 2)
    CONV_CASE(16, 1)
#undef CONV_CASE
    return OF_ERR_UNSUPPORTED;
}

int wgrad_tiles(int B, int H, int W) { return B * ((H + kWgRows - 1) / kWgRows) * ((W + 7) / 8); }

int launch_wgrad(const float* dY, int N, const float* X, int CX, int B, int H, int W, int Kpad, int blocks,
                 float* part, float* bpart, hipStream_t st)
{
    const int ntiles = wgrad_tiles(B, H, W);
#define WG_CASE(cx, n)                                                                                 \
    if (CX == cx && N == n) {                                                                          \
        hipLaunchKernelGGL((k_wgrad<cx, n>), dim3(blocks), dim3(256), 0, st, dY, X, B, H, W, ntiles, \
                           Kpad, part, bpart);                                                 \
        CNN_CHECK("k_wgrad");                                                                          \
        return OF_OK;                                                                                  \
    }
    WG_CASE(5, 32)
    WG_CASE(32, 32)
    WG_CASE(32, 2)
#undef WG_CASE
    return OF_ERR_UNSUPPORTED;
}

struct Layer {
    int cin = 0, cout = 0, relu = 0;
    size_t woff = 0, boff = 0;   // offsets into the parameter vector
    int Kpad = 0, Npad = 0, Cpad = 0;   // Kpad: 9*cin padded, the row of the weight-gradient partials
    short* fwd = nullptr;        // bf16 packs
    short* bwd = nullptr;
};

}  // namespace
}  // namespace amdflow

using namespace amdflow;

struct of_cnn {
    int hidden = 0, channels = 0;
    std::vector<Layer> layers;
    size_t nparams = 0;
    float* w = nullptr;   // fp32 master weights: per layer W[n][t][c], then bias[n]
    float* g = nullptr;
    float* m = nullptr;
    float* v = nullptr;
    int step = 0;
    // batch workspace, grown on demand
    long long cap_px = 0;
    std::vector<float*> act;   // output of every layer, NHWC
    float* dA = nullptr;       // gradient ping-pong buffers
    float* dB = nullptr;
    float* part = nullptr;     // weight / bias gradient partials
    double* lpart = nullptr;   // loss partials
    double* loss = nullptr;
    // single-image inference workspace
    long long cap_in = 0;
    float* xin = nullptr;      // 5-channel features
    float* pred = nullptr;     // planar prediction
    // warm-start workspace: the prediction carried to the first solved scale, zero flow
    long long cap_lift = 0;
    float* lift = nullptr;
    float* zero = nullptr;
};

namespace {

constexpr int kLossBlocks = 1024;

void free_ws(of_cnn* h)
{
    for (float*& p : h->act) dev_free(p);
    h->act.clear();
    dev_free(h->dA);
    dev_free(h->dB);
    dev_free(h->part);
    h->cap_px = 0;
}

int ensure_ws(of_cnn* h, long long px)
{
    if (px <= h->cap_px) return OF_OK;
    OF_HIP(hipDeviceSynchronize());   // queued work may still use the old buffers
    free_ws(h);
    int maxc = 5;
    size_t need = 1;
    const size_t blocks = (size_t)std::min<long long>(kWgMaxBlocks, px);   // a tile holds a pixel at least
    for (const Layer& L : h->layers) {
        float* p = nullptr;
        OF_TRY(dev_alloc(&p, (size_t)px * L.cout));
        h->act.push_back(p);
        maxc = std::max(maxc, std::max(L.cin, L.cout));
        need = std::max(need, blocks * (size_t)(L.Npad * L.Kpad + L.cout));
    }
    OF_TRY(dev_alloc(&h->dA, (size_t)px * maxc));
    OF_TRY(dev_alloc(&h->dB, (size_t)px * maxc));
    OF_TRY(dev_alloc(&h->part, need));
    h->cap_px = px;
    return OF_OK;
}

int ensure_in(of_cnn* h, long long n)
{
    if (n <= h->cap_in) return OF_OK;
    OF_HIP(hipDeviceSynchronize());
    dev_free(h->xin);
    dev_free(h->pred);
    h->cap_in = 0;
    OF_TRY(dev_alloc(&h->xin, (size_t)n * 5));
    OF_TRY(dev_alloc(&h->pred, (size_t)n * 2));
    h->cap_in = n;
    return OF_OK;
}

int pack(of_cnn* h, hipStream_t st)
{
    for (Layer& L : h->layers) {
        const int n = std::max(L.Npad * pad_k(L.cin), L.Cpad * pad_k(L.cout));
        hipLaunchKernelGGL(k_pack, dim3(blocks256(n)), dim3(256), 0, st, h->w + L.woff, L.cout, L.cin,
                           L.Npad, L.Cpad, L.fwd, L.bwd);
        CNN_CHECK("k_pack");
    }
    return OF_OK;
}

// The network's layers; the last one writes `Y`, or its activation buffer if
// that is null.
int forward(of_cnn* h, const float* X, int B, int H, int W, float* Y, hipStream_t st)
{
    const float* in = X;
    for (size_t l = 0; l < h->layers.size(); l++) {
        const Layer& L = h->layers[l];
        float* out = Y && l + 1 == h->layers.size() ? Y : h->act[l];
        OF_TRY(launch_conv(in, B, H, W, L.cin, L.fwd, L.cout, h->w + L.boff, 1, L.relu,
                           nullptr, out, st));
        in = out;
    }
    return OF_OK;
}

// Backward pass from the loss gradient in h->dA; fills h->g.
int backward(of_cnn* h, const float* X, int B, int H, int W, hipStream_t st)
{
    const int blocks = std::min(kWgMaxBlocks, wgrad_tiles(B, H, W));
    float* dcur = h->dA;
    float* dnext = h->dB;
    for (int l = (int)h->layers.size() - 1; l >= 0; l--) {
        const Layer& L = h->layers[l];
        const float* in = l ? h->act[l - 1] : X;
        const int K = 9 * L.cin;
        float* bpart = h->part + (size_t)blocks * L.Npad * L.Kpad;
        OF_TRY(launch_wgrad(dcur, L.cout, in, L.cin, B, H, W, L.Kpad, blocks, h->part, bpart, st));
        hipLaunchKernelGGL(k_grad_reduce, dim3((L.cout * (K + 1) + 63) / 64), dim3(1024), 0, st, h->part,
                           blocks, L.Npad, L.Kpad, L.cout, K, h->g + L.woff, bpart, h->g + L.boff);
        CNN_CHECK("k_grad_reduce");
        if (l == 0) break;
        // gradient w.r.t. this layer's input, zero where the ReLU below was inactive
        const Layer& P = h->layers[l - 1];
        OF_TRY(launch_conv(dcur, B, H, W, L.cout, L.bwd, L.cin, nullptr, -1, 0,
                           P.relu ? h->act[l - 1] : nullptr, dnext, st));
        std::swap(dcur, dnext);
    }
    return OF_OK;
}

int loss_grad(of_cnn* h, const float* T, int B, int H, int W, hipStream_t st)
{
    const long long M = (long long)B * H * W;
    const unsigned blocks = std::min<unsigned>(kLossBlocks, blocks256(2 * M));
    hipLaunchKernelGGL(k_mse, dim3(blocks), dim3(256), 0, st, h->act.back(), T, M, H * W,
                       1.0f / (float)M, h->dA, h->lpart);
    CNN_CHECK("k_mse");
    hipLaunchKernelGGL(k_sum_f64, dim3(1), dim3(256), 0, st, h->lpart, (int)blocks, 0.5 / (double)M, h->loss);
    CNN_CHECK("k_sum_f64");
    return OF_OK;
}

void release(of_cnn* h)
{
    if (!h) return;
    free_ws(h);
    for (Layer& L : h->layers) {
        dev_free(L.fwd);
        dev_free(L.bwd);
    }
    dev_free(h->w);
    dev_free(h->g);
    dev_free(h->m);
    dev_free(h->v);
    dev_free(h->lpart);
    dev_free(h->loss);
    dev_free(h->xin);
    dev_free(h->pred);
    dev_free(h->lift);
    dev_free(h->zero);
    delete h;
}

bool dims_ok(const of_cnn* h, const void* a, const void* b, int B, int H, int W)
{
    return h && a && b && B >= 1 && H >= 1 && W >= 1 && (long long)B * H * W < (1ll << 31) / 64;
}

}  // namespace

extern "C" {

int of_cnn_create(int hidden_layers, int channels, unsigned long long seed, of_cnn** out)
{
    return guarded([&]() -> int {
        if (!out) return OF_ERR_ARG;
        *out = nullptr;
        if (hidden_layers < 0 || hidden_layers > 16 || channels != 32) return OF_ERR_ARG;
        of_cnn* h = new (std::nothrow) of_cnn();
        if (!h) return OF_ERR_ALLOC;
        h->hidden = hidden_layers;
        h->channels = channels;
        std::vector<std::pair<int, int>> dims;
        dims.push_back({5, channels});
        for (int i = 0; i < hidden_layers; i++) dims.push_back({channels, channels});
        dims.push_back({channels, 2});
        size_t off = 0;
        for (size_t i = 0; i < dims.size(); i++) {
            Layer L;
            L.cin = dims[i].first;
            L.cout = dims[i].second;
            L.relu = i + 1 < dims.size();
            L.woff = off;
            off += (size_t)L.cout * 9 * L.cin;
            L.boff = off;
            off += L.cout;
            L.Kpad = pad32(9 * L.cin);
            L.Npad = pad16(L.cout);
            L.Cpad = pad16(L.cin);
            h->layers.push_back(L);
        }
        h->nparams = off;
        // He-normal initial weights (the head scaled by 0.1), zero biases
        std::vector<float> w(off, 0.0f);
        std::mt19937_64 rng(seed);
        for (const Layer& L : h->layers) {
            const float sd = std::sqrt(2.0f / (9.0f * (float)L.cin)) * (L.relu ? 1.0f : 0.1f);
            std::normal_distribution<float> nd(0.0f, sd);
            for (size_t i = 0; i < (size_t)L.cout * 9 * L.cin; i++) w[L.woff + i] = nd(rng);
        }
        int st = dev_alloc(&h->w, off);
        if (!st) st = dev_alloc(&h->g, off);
        if (!st) st = dev_alloc(&h->m, off);
        if (!st) st = dev_alloc(&h->v, off);
        if (!st) st = dev_alloc(&h->lpart, kLossBlocks);
        if (!st) st = dev_alloc(&h->loss, 1);
        for (Layer& L : h->layers) {
            if (!st) st = dev_alloc(&L.fwd, (size_t)L.Npad * pad_k(L.cin));
            if (!st) st = dev_alloc(&L.bwd, (size_t)L.Cpad * pad_k(L.cout));
        }
        if (!st && hipMemcpy(h->w, w.data(), off * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) st = OF_ERR_HIP;
        if (!st && hipMemset(h->g, 0, off * sizeof(float)) != hipSuccess) st = OF_ERR_HIP;
        if (!st && hipMemset(h->m, 0, off * sizeof(float)) != hipSuccess) st = OF_ERR_HIP;
        if (!st && hipMemset(h->v, 0, off * sizeof(float)) != hipSuccess) st = OF_ERR_HIP;
        if (!st) st = pack(h, nullptr);
        if (!st && hipDeviceSynchronize() != hipSuccess) st = OF_ERR_HIP;
        if (st) {
            (void)hipGetLastError();
            release(h);
            return st;
        }
        *out = h;
        return OF_OK;
    });
}

void of_cnn_destroy(of_cnn* h) { release(h); }

long long of_cnn_num_params(const of_cnn* h) { return h ? (long long)h->nparams : 0; }

int of_cnn_get_params(const of_cnn* h, float* host)
{
    if (!h || !host) return OF_ERR_ARG;
    OF_HIP(hipDeviceSynchronize());
    OF_HIP(hipMemcpy(host, h->w, h->nparams * sizeof(float), hipMemcpyDeviceToHost));
    return OF_OK;
}

int of_cnn_set_params(of_cnn* h, const float* host)
{
    if (!h || !host) return OF_ERR_ARG;
    OF_HIP(hipDeviceSynchronize());
    OF_HIP(hipMemcpy(h->w, host, h->nparams * sizeof(float), hipMemcpyHostToDevice));
    OF_HIP(hipMemset(h->m, 0, h->nparams * sizeof(float)));
    OF_HIP(hipMemset(h->v, 0, h->nparams * sizeof(float)));
    h->step = 0;
    OF_TRY(pack(h, nullptr));
    OF_HIP(hipDeviceSynchronize());
    return OF_OK;
}

int of_cnn_features(const float* dI0s, const float* dI1s, int H, int W, float* dX, void* stream)
{
    if (!dI0s || !dI1s || !dX || H < 1 || W < 1 || (long long)H * W >= (1ll << 31) / 8) return OF_ERR_ARG;
    hipLaunchKernelGGL(k_features, dim3(blocks256((long long)H * W)), dim3(256), 0, (hipStream_t)stream,
                       dI0s, dI1s, H, W, dX);
    CNN_CHECK("k_features");
    return OF_OK;
}

int of_cnn_forward(of_cnn* h, const float* dX, int B, int H, int W, float* dY, void* stream)
{
    return guarded([&]() -> int {
        if (!dims_ok(h, dX, dY, B, H, W)) return OF_ERR_ARG;
        hipStream_t st = (hipStream_t)stream;
        OF_TRY(ensure_ws(h, (long long)B * H * W));
        return forward(h, dX, B, H, W, dY, st);
    });
}

int of_cnn_predict(of_cnn* h, const float* dI0s, const float* dI1s, int H, int W, float* dU, void* stream)
{
    return guarded([&]() -> int {
        if (!dims_ok(h, dI0s, dI1s, 1, H, W) || !dU) return OF_ERR_ARG;
        hipStream_t st = (hipStream_t)stream;
        const long long n = (long long)H * W;
        OF_TRY(ensure_in(h, n));
        OF_TRY(ensure_ws(h, n));
        OF_TRY(of_cnn_features(dI0s, dI1s, H, W, h->xin, st));
        OF_TRY(forward(h, h->xin, 1, H, W, nullptr, st));
        hipLaunchKernelGGL(k_to_planar, dim3(blocks256(n)), dim3(256), 0, st, h->act.back(), (int)n, dU);
        CNN_CHECK("k_to_planar");
        return OF_OK;
    });
}

int of_cnn_gradients(of_cnn* h, const float* dX, const float* dT, int B, int H, int W, float* host_grads,
                     double* loss)
{
    return guarded([&]() -> int {
        if (!dims_ok(h, dX, dT, B, H, W)) return OF_ERR_ARG;
        OF_TRY(ensure_ws(h, (long long)B * H * W));
        OF_TRY(forward(h, dX, B, H, W, nullptr, nullptr));
        OF_TRY(loss_grad(h, dT, B, H, W, nullptr));
        OF_TRY(backward(h, dX, B, H, W, nullptr));
        OF_HIP(hipDeviceSynchronize());
        if (host_grads) OF_HIP(hipMemcpy(host_grads, h->g, h->nparams * sizeof(float), hipMemcpyDeviceToHost));
        if (loss) OF_HIP(hipMemcpy(loss, h->loss, sizeof(double), hipMemcpyDeviceToHost));
        return OF_OK;
    });
}

int of_cnn_train_step(of_cnn* h, const float* dX, const float* dT, int B, int H, int W, float lr,
                      double* loss)
{
    return guarded([&]() -> int {
        if (!dims_ok(h, dX, dT, B, H, W) || !(lr > 0.0f)) return OF_ERR_ARG;
        OF_TRY(ensure_ws(h, (long long)B * H * W));
        OF_TRY(forward(h, dX, B, H, W, nullptr, nullptr));
        OF_TRY(loss_grad(h, dT, B, H, W, nullptr));
        OF_TRY(backward(h, dX, B, H, W, nullptr));
        h->step++;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.0f - std::pow(b1, (float)h->step), c2 = 1.0f - std::pow(b2, (float)h->step);
        hipLaunchKernelGGL(k_adam, dim3(blocks256((long long)h->nparams)), dim3(256), 0, nullptr, h->w, h->g,
                           h->m, h->v, (int)h->nparams, lr, b1, b2, 1e-8f, c1, c2);
        CNN_CHECK("k_adam");
        OF_TRY(pack(h, nullptr));
        if (loss) OF_HIP(hipMemcpy(loss, h->loss, sizeof(double), hipMemcpyDeviceToHost));
        else OF_HIP(hipDeviceSynchronize());
        return OF_OK;
    });
}

// Warm-started solve of one pair: prepare the pyramids, predict the
// coarsest-scale flow, carry it to `first_scale`, keep it only if its TV-L1
// energy there is not above that of zero flow, then solve scales
// first_scale .. 0 with at most `warps` warpings and `max_iterations`
// iterations per warping (0: the handle's parameters).  When zero flow wins,
// the solve is the plain one: zero initial flow at the coarsest scale and
// the handle's own parameters.
int of_tvl1_warm_run_device_u8(of_tvl1* tv, of_cnn* net, const uint8_t* dI0, const uint8_t* dI1,
                               int first_scale, int warps, int max_iterations, float* dU,
                               int* fell_back, double* energies, void* stream)
{
    return guarded([&]() -> int {
        if (!tv || !net || !dI0 || !dI1 || !dU || warps < 0 || max_iterations < 0) return OF_ERR_ARG;
        const int ns = of_tvl1_nscales(tv);
        if (first_scale < -1 || first_scale >= ns) return OF_ERR_ARG;
        if (first_scale < 0) first_scale = ns - 1;
        int nx = 0, ny = 0, fx = 0, fy = 0;
        OF_TRY(of_tvl1_scale_size(tv, ns - 1, &nx, &ny));
        OF_TRY(of_tvl1_scale_size(tv, first_scale, &fx, &fy));
        const long long n = (long long)nx * ny, nf = (long long)fx * fy;
        OF_TRY(ensure_in(net, n));
        if (2 * nf > net->cap_lift) {
            OF_HIP(hipDeviceSynchronize());
            dev_free(net->lift);
            dev_free(net->zero);
            net->cap_lift = 0;
            OF_TRY(dev_alloc(&net->lift, 2 * (size_t)nf));
            OF_TRY(dev_alloc(&net->zero, 2 * (size_t)nf));
            net->cap_lift = 2 * nf;
        }
        hipStream_t st = (hipStream_t)stream;
        OF_TRY(of_tvl1_prepare_device_u8(tv, dI0, dI1, stream));
        const float* I0c = nullptr;
        const float* I1c = nullptr;
        OF_TRY(of_tvl1_scale_images(tv, ns - 1, &I0c, &I1c));
        OF_TRY(of_cnn_predict(net, I0c, I1c, ny, nx, net->pred, stream));
        OF_TRY(of_tvl1_lift_flow(tv, ns - 1, net->pred, first_scale, net->lift, stream));
        OF_HIP(hipMemsetAsync(net->zero, 0, sizeof(float) * 2 * (size_t)nf, st));
        double ep[3], ez[3];
        OF_TRY(of_tvl1_energy(tv, first_scale, net->lift, ep, stream));
        OF_TRY(of_tvl1_energy(tv, first_scale, net->zero, ez, stream));
        if (energies) {
            energies[0] = ep[0];
            energies[1] = ez[0];
        }
        const bool keep = ep[0] <= ez[0];
        if (fell_back) *fell_back = keep ? 0 : 1;
        if (keep) return of_tvl1_solve_prepared(tv, net->lift, first_scale, warps, max_iterations, dU, stream);
        return of_tvl1_solve_prepared(tv, nullptr, -1, 0, 0, dU, stream);
    });
}

// ---- test entry point: MFMA operand layout through k_conv_lds ----

// D = A (16x16) * B (16x16), row-major fp32 (operands rounded to bf16),
// computed as a convolution of a 1x16 image with 16 channels whose only
// non-zero tap is the centre one.
int of_dbg_cnn_mfma(const float* A, const float* Bm, float* D)
{
    return guarded([&]() -> int {
        if (!A || !Bm || !D) return OF_ERR_ARG;
        float* dX = nullptr;
        float* dY = nullptr;
        short* dW = nullptr;
        const int Kpad = pad_k(16);
        int st = dev_alloc(&dX, 256);
        if (!st) st = dev_alloc(&dY, 256);
        if (!st) st = dev_alloc(&dW, 16 * Kpad);
        std::vector<short> w(16 * Kpad, 0);
        for (int n = 0; n < 16; n++)
            for (int c = 0; c < 16; c++) w[n * Kpad + 4 * 16 + c] = to_bf16(Bm[c * 16 + n]);
        if (!st && hipMemcpy(dX, A, 256 * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) st = OF_ERR_HIP;
        if (!st && hipMemcpy(dW, w.data(), w.size() * sizeof(short), hipMemcpyHostToDevice) != hipSuccess)
            st = OF_ERR_HIP;
        if (!st) st = launch_conv(dX, 1, 1, 16, 16, dW, 16, nullptr, 1, 0, nullptr, dY, nullptr);
        if (!st && hipDeviceSynchronize() != hipSuccess) st = OF_ERR_HIP;
        if (!st && hipMemcpy(D, dY, 256 * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) st = OF_ERR_HIP;
        dev_free(dX);
        dev_free(dY);
        dev_free(dW);
        return st;
    });
}

}  // extern "C"
