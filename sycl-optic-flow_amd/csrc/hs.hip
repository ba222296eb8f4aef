// hs.hip -- Horn-Schunck on gfx950: kernels, host orchestration and C ABI.
//
// Follows the control flow of ComputeFlow (src/hs/cuda/flow.cu:112-208):
// a /2 pyramid, coarse to fine, nWarpIters x (warp I1, derivatives,
// nSolverIters Jacobi sweeps, u += du), flow upscaled between levels.  The
// reference kernels index images incorrectly (warpingKernel.cuh:38-42,
// upscaleKernel.cuh:33-39, derivativesKernel.cuh:42-46); these kernels
// implement what they intend: bilinear sampling with clamp-to-edge
// addressing and clamp-to-edge stencils.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <new>

#include "amdflow.h"
#include "amdflow_debug.h"
#include "common.hpp"
#include "device_math.hpp"

namespace amdflow {
namespace {

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// Bilinear sample at (x, y) in pixel-centre coordinates, clamp-to-edge.
__device__ __forceinline__ float bilinear_at(const float* __restrict__ src, int w, int h, int s,
                                             float x, float y)
{
    const float fx0 = floorf(x), fy0 = floorf(y);
    const float ax = x - fx0, ay = y - fy0;
    // limited to [-1, w] first so that +1 cannot overflow (clamps unchanged)
    const int x0 = clampi(f2i_sat(fx0), -1, w), y0 = clampi(f2i_sat(fy0), -1, h);
    const int xa = clampi(x0, 0, w - 1), xb = clampi(x0 + 1, 0, w - 1);
    const int ya = clampi(y0, 0, h - 1), yb = clampi(y0 + 1, 0, h - 1);
    const float a = src[(size_t)ya * s + xa], b = src[(size_t)ya * s + xb];
    const float c = src[(size_t)yb * s + xa], d = src[(size_t)yb * s + xb];
    const float top = (1.0f - ax) * a + ax * b;
    const float bot = (1.0f - ax) * c + ax * d;
    return (1.0f - ay) * top + ay * bot;
}

// 2x2 box average (downscaleKernel.cuh:27-40), every output pixel.
__global__ __launch_bounds__(256) void k_hs_downscale(const float* __restrict__ src, int s,
                                                      float* __restrict__ out, int nw, int nh,
                                                      int ns)
{
    const int ix = blockIdx.x * 64 + (threadIdx.x & 63);
    const int iy = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (ix >= nw || iy >= nh) return;
    const size_t sx = (size_t)ix * 2, sy = (size_t)iy * 2;
    const float a = src[sx + sy * s], b = src[sx + (sy + 1) * s];
    const float c = src[(sx + 1) + sy * s], d = src[(sx + 1) + (sy + 1) * s];
    out[(size_t)ix + (size_t)iy * ns] = 0.25f * (((a + b) + c) + d);
}

// Flow upscale x2 at ((ix-0.5)/2, (iy-0.5)/2) times `scale`
// (upscaleKernel.cuh:26-40).
__global__ __launch_bounds__(256) void k_hs_upscale(const float* __restrict__ src, int w, int h,
                                                    int s, float* __restrict__ out, int nw, int nh,
                                                    int ns, float scale)
{
    const int ix = blockIdx.x * 64 + (threadIdx.x & 63);
    const int iy = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (ix >= nw || iy >= nh) return;
    const float x = ((float)ix - 0.5f) * 0.5f;
    const float y = ((float)iy - 0.5f) * 0.5f;
    out[(size_t)ix + (size_t)iy * ns] = bilinear_at(src, w, h, s, x, y) * scale;
}

// Warp I1 by (u, v) then the derivatives of derivativesKernel.cuh:29-73:
// 5-tap [1 -8 0 8 -1]/12 on I0 and on the warped I1 (clamp to edge),
// Ix/Iy = mean of the two, Iz = I1w - I0.  The warped image is computed at
// the 9 stencil positions it is needed at.
__device__ __forceinline__ float d5(float m2, float m1, float p1, float p2)
{
    float t = m2;
    t -= m1 * 8.0f;
    t += p1 * 8.0f;
    t -= p2;
    t /= 12.0f;
    return t;
}

// Tile of the fused warp + derivatives kernel: kWdX x kWdY output pixels per
// workgroup, the warped frame staged in LDS with the stencil's 2-pixel halo.
constexpr int kWdX = 64, kWdY = 8, kWdH = 2;

// Warp and derivatives in one launch: the workgroup warps its tile plus halo
// into LDS (a halo position takes the clamped pixel's warp, which is what the
// clamped stencil reads), then every thread forms the derivatives of two
// pixels from LDS and I0.  A launch costs about as much as its memory traffic
// at these sizes; one launch instead of two also drops the round trip of the
// warped plane (1280x720: 3.2 + 3.5 us before).
__global__ __launch_bounds__(256) void k_hs_warp_derivs(const float* __restrict__ I0,
                                                        const float* __restrict__ I1, int w, int h,
                                                        int s, const float* __restrict__ u,
                                                        const float* __restrict__ v,
                                                        float* __restrict__ Ix,
                                                        float* __restrict__ Iy,
                                                        float* __restrict__ Iz,
                                                        float* __restrict__ I1w_out)
{
    constexpr int PX = kWdX + 2 * kWdH, PY = kWdY + 2 * kWdH;
    __shared__ float sw[PY][PX];
    const int x0 = blockIdx.x * kWdX, y0 = blockIdx.y * kWdY;
    for (int e = threadIdx.x; e < PX * PY; e += 256) {
        const int py = e / PX, px = e - py * PX;
        const int ix = clampi(x0 + px - kWdH, 0, w - 1), iy = clampi(y0 + py - kWdH, 0, h - 1);
        const size_t pos = (size_t)ix + (size_t)iy * s;
        sw[py][px] = bilinear_at(I1, w, h, s, (float)ix + u[pos], (float)iy + v[pos]);
    }
    __syncthreads();
    const int lx = threadIdx.x & 63;
    const int ix = x0 + lx;
    if (ix >= w) return;
    const int xm2 = clampi(ix - 2, 0, w - 1), xm1 = clampi(ix - 1, 0, w - 1);
    const int xp1 = clampi(ix + 1, 0, w - 1), xp2 = clampi(ix + 2, 0, w - 1);
#pragma unroll
    for (int k = 0; k < kWdY / 4; k++) {
        const int ly = (threadIdx.x >> 6) + 4 * k;
        const int iy = y0 + ly;
        if (iy >= h) return;
        const size_t row = (size_t)iy * s, pos = row + ix;
        const size_t ym2 = (size_t)clampi(iy - 2, 0, h - 1) * s, ym1 = (size_t)clampi(iy - 1, 0, h - 1) * s;
        const size_t yp1 = (size_t)clampi(iy + 1, 0, h - 1) * s, yp2 = (size_t)clampi(iy + 2, 0, h - 1) * s;
        const float* c = &sw[ly + kWdH][lx + kWdH];
        const float t0 = d5(I0[row + xm2], I0[row + xm1], I0[row + xp1], I0[row + xp2]);
        const float t1 = d5(c[-2], c[-1], c[1], c[2]);
        Ix[pos] = (t0 + t1) * 0.5f;
        Iz[pos] = c[0] - I0[pos];
        const float r0 = d5(I0[ym2 + ix], I0[ym1 + ix], I0[yp1 + ix], I0[yp2 + ix]);
        const float r1 = d5(c[-2 * PX], c[-PX], c[PX], c[2 * PX]);
        Iy[pos] = (r0 + r1) * 0.5f;
        if (I1w_out) I1w_out[pos] = c[0];
    }
}

// One launch of Jacobi sweeps (solverKernel.cuh:39-153): `kk` sweeps (at most
// the halo K) of every pixel.
struct JacobiArgs {
    const float *du0, *dv0;        // input increments
    const float *Ix, *Iy, *Iz;
    float *du1, *dv1;              // output increments; unused with `u` set
    float *u, *v;                  // set on a warping's last launch: u += du, v += dv
    int w, h, s;
    float alpha;
    int K, kk;
    int zero_in;                   // the input increments are all zero
};

// 1/d of a float in double, to about an ulp: the hardware reciprocal and two
// Newton steps.  0, infinite and NaN divisors give garbage (div_by fixes it).
__device__ __forceinline__ double recip_f64(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
    return __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
}

// The IEEE float quotient n / d from d's double reciprocal y = recip_f64(d),
// for a divisor that stays while the numerators change: 6 instructions
// instead of the 11 of the division sequence.  The corrected double quotient
// is exact where n / d has at most 53 bits (so also on every float rounding
// boundary, subnormal ones included) and otherwise within 2^-52 of n / d,
// which is never within 2^-49 of a boundary: rounding it gives the IEEE
// quotient.  v_div_fixup supplies the special values.
__device__ __forceinline__ float div_by(float n, float d, double dd, double y)
{
    const double nd = (double)n;
    double q = nd * y;
    q = __builtin_fma(__builtin_fma(-q, dd, nd), y, q);
    return __builtin_amdgcn_div_fixupf((float)q, d, n);
}

// K sweeps per launch (the halo) on tiles of 64 columns (one per lane) by
// NW*R rows (R consecutive rows per wave, in registers); horizontal
// neighbours by lane shifts, vertical ones from registers or one LDS row per
// wave (double-buffered: one barrier per sweep).  Values within K pixels of
// the tile edge go stale one pixel per sweep; the central (64-2K) x (NW*R-2K)
// pixels are stored.
// Left and right of the image the tile holds the mirrored columns.  They stay
// the mirror image sweep after sweep (left + right commutes bit for bit), so
// the neighbour across the border is the clamped one without a select.  Up
// and down do not commute in the sum: tiles that reach the first or last row
// (EDGE) take selects there.
template <int R, int NW, bool EDGE>
__device__ __forceinline__ void jacobi_tile(const JacobiArgs& a, float (*sh)[4][NW][64])
{
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int w = a.w, h = a.h, K = a.K;
    const int TW = 64 - 2 * K, TH = NW * R - 2 * K;
    const int x = (int)blockIdx.x * TW - K + lane;
    const int oy0 = (int)blockIdx.y * TH;
    const int ybase = oy0 - K + wave * R;
    int xm = x;
    if (xm < 0 || xm >= w) {
        xm %= 2 * w;
        if (xm < 0) xm += 2 * w;
        if (xm >= w) xm = 2 * w - 1 - xm;
    }

    float u[R], v[R], gx[R], gy[R], gz[R], den[R];
    double dd[R], rd[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int y = ybase + r;
        u[r] = v[r] = gx[r] = gy[r] = gz[r] = 0.0f;
        if (!EDGE || (y >= 0 && y < h)) {
            const size_t p = (size_t)y * a.s + xm;
            gx[r] = a.Ix[p];
            gy[r] = a.Iy[p];
            gz[r] = a.Iz[p];
            if (!a.zero_in) {
                u[r] = a.du0[p];
                v[r] = a.dv0[p];
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        den[r] = (gx[r] * gx[r] + gy[r] * gy[r]) + a.alpha;
        dd[r] = (double)den[r];
        rd[r] = recip_f64(dd[r]);
    }

    // the outermost waves read their own rows: stale, never stored
    const int wu = wave < NW - 1 ? wave + 1 : wave, wd = wave ? wave - 1 : wave;
    auto sweep = [&](float(*b)[NW][64]) {
        b[0][wave][lane] = u[0];
        b[1][wave][lane] = v[0];
        b[2][wave][lane] = u[R - 1];
        b[3][wave][lane] = v[R - 1];
        // left + right of every row while the LDS rows travel
        float hu[R], hv[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            hu[r] = lane_left(u[r]) + lane_right(u[r]);
            hv[r] = lane_left(v[r]) + lane_right(v[r]);
        }
        __syncthreads();
        const float upU = b[0][wu][lane], upV = b[1][wu][lane];
        float du = b[2][wd][lane], dv = b[3][wd][lane];
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int y = ybase + r;
            const bool top = EDGE && y <= 0, bottom = EDGE && y >= h - 1;
            const float cu = u[r], cv = v[r];
            const float uu = r < R - 1 ? u[r + 1] : upU, uv = r < R - 1 ? v[r + 1] : upV;
            // "up" is row y+1 and "down" row y-1, clamped at the image edge
            const float sumU = ((hu[r] + (bottom ? cu : uu)) + (top ? cu : du)) * 0.25f;
            const float sumV = ((hv[r] + (bottom ? cv : uv)) + (top ? cv : dv)) * 0.25f;
            const float frac = div_by((gx[r] * sumU + gy[r] * sumV) + gz[r], den[r], dd[r], rd[r]);
            u[r] = sumU - gx[r] * frac;
            v[r] = sumV - gy[r] * frac;
            du = cu;
            dv = cv;
        }
    };
    // two sweeps per trip: the LDS buffer of each is known at compile time
#pragma unroll 1
    for (int t = 0; t < a.kk; t += 2) {
        sweep(sh[0]);
        if (t + 1 < a.kk) sweep(sh[1]);
    }
    if (!(x >= 0 && x < w && lane >= K && lane < K + TW)) return;
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int y = ybase + r;
        if (y >= oy0 && y < oy0 + TH && (!EDGE || y < h)) {
            const size_t p = (size_t)y * a.s + x;
            if (a.u) {
                a.u[p] = a.u[p] + u[r];
                a.v[p] = a.v[p] + v[r];
            } else {
                a.du1[p] = u[r];
                a.dv1[p] = v[r];
            }
        }
    }
}

template <int R, int NW>
__global__ __launch_bounds__(64 * NW) void k_hs_jacobi(JacobiArgs a)
{
    __shared__ float sh[2][4][NW][64];   // [buffer][first u, first v, last u, last v][wave][lane]
    const int y0 = (int)blockIdx.y * (NW * R - 2 * a.K) - a.K;
    if (y0 >= 1 && y0 + NW * R - 1 <= a.h - 2) jacobi_tile<R, NW, false>(a, sh);
    else jacobi_tile<R, NW, true>(a, sh);
}

// Frames in and flow cleared, or flow out: two planes of n floats copied and
// two of nz cleared, in one launch.
__global__ __launch_bounds__(256) void k_hs_copy2(const float* a0, float* a1, const float* b0, float* b1,
                                                  size_t n, float* z0, float* z1, size_t nz)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n || i < nz;
         i += (size_t)gridDim.x * blockDim.x) {
        if (i < n) {
            a1[i] = a0[i];
            b1[i] = b0[i];
        }
        if (i < nz) z0[i] = z1[i] = 0.0f;
    }
}

inline dim3 grid2d(int w, int h) { return dim3(cdiv(w, 64), cdiv(h, 4)); }

#define HS_CHECK(name)                                      \
    do {                                                    \
        hipError_t e_ = hipGetLastError();                  \
        if (e_ != hipSuccess) {                             \
            record_hip_error(e_, name, __FILE__, __LINE__); \
            return OF_ERR_HIP;                              \
        }                                                   \
    } while (0)

// Waves per workgroup of the shapes set by of_hs_set_jacobi_shape: 64 x 8R
// pixel tiles.
constexpr int kHsWaves = 8;

bool jacobi_shape_ok(int K, int R)
{
    if (!(K == 1 || K == 2 || K == 4 || K == 8)) return false;
    if (!(R == 2 || R == 4 || R == 8)) return false;
    return kHsWaves * R - 2 * K >= 4;
}

// A launch shape: sweeps per launch (the halo), rows per wave, waves.
struct JacobiShape {
    int K, R, NW;
};

template <int R, int NW>
int launch_jacobi_rn(const JacobiArgs& a, hipStream_t st)
{
    const dim3 g(cdiv(a.w, 64 - 2 * a.K), cdiv(a.h, NW * R - 2 * a.K));
    hipLaunchKernelGGL((k_hs_jacobi<R, NW>), g, dim3(64 * NW), 0, st, a);
    HS_CHECK("k_hs_jacobi");
    return OF_OK;
}

int launch_jacobi(const JacobiShape& t, const JacobiArgs& a, hipStream_t st)
{
    if (t.K < 1 || 2 * t.K >= 64 || 2 * t.K >= t.R * t.NW || a.kk > t.K) return OF_ERR_ARG;
#define HS_CASE(r, n) \
    if (t.R == r && t.NW == n) return launch_jacobi_rn<r, n>(a, st);
    HS_CASE(2, 8) HS_CASE(4, 8) HS_CASE(8, 8) HS_CASE(2, 16) HS_CASE(3, 16)
#undef HS_CASE
    return OF_ERR_UNSUPPORTED;
}

// n Jacobi sweeps from (du0,dv0) (or from zero).  With u/v the last launch
// adds the increments to them; otherwise *result names the buffer holding
// the result (0: du[0]/dv[0], 1: du[1]/dv[1]).
int run_jacobi(const JacobiShape& t, JacobiArgs a, float* du[2], float* dv[2], int n, bool zero_first,
               float* u, float* v, int* result, hipStream_t st)
{
    int cur = 0;
    a.K = t.K;
    a.zero_in = zero_first ? 1 : 0;
    for (int done = 0; done < n;) {
        a.kk = (n - done) < t.K ? (n - done) : t.K;
        done += a.kk;
        a.du0 = du[cur];
        a.dv0 = dv[cur];
        a.du1 = du[cur ^ 1];
        a.dv1 = dv[cur ^ 1];
        a.u = done == n ? u : nullptr;
        a.v = done == n ? v : nullptr;
        OF_TRY(launch_jacobi(t, a, st));
        a.zero_in = 0;
        cur ^= 1;
    }
    *result = cur;
    return OF_OK;
}

}  // namespace
}  // namespace amdflow

using namespace amdflow;

struct of_hs {
    int nLevels = 0, stride = 0, W = 0, H = 0;
    hipStream_t stream = nullptr;
    float** pI0 = nullptr;
    float** pI1 = nullptr;
    int pW[32]{}, pH[32]{}, pS[32]{};
    size_t plane = 0;   // floats of the largest level's plane: of each buffer from u to Iz
    float *u = nullptr, *v = nullptr, *nu = nullptr, *nv = nullptr;
    float *du[2]{}, *dv[2]{};
    float *Ix = nullptr, *Iy = nullptr, *Iz = nullptr;
    float *hin0 = nullptr, *hin1 = nullptr;   // device staging of host inputs
    int K = 0, R = 0;                         // Jacobi launch shape set by the caller; 0: by frame size
};

namespace {

void hs_release(of_hs* h)
{
    if (!h) return;
    for (int l = 0; l < h->nLevels; l++) {
        if (h->pI0) dev_free(h->pI0[l]);
        if (h->pI1) dev_free(h->pI1[l]);
    }
    delete[] h->pI0;
    delete[] h->pI1;
    dev_free(h->u); dev_free(h->v); dev_free(h->nu); dev_free(h->nv);
    dev_free(h->du[0]); dev_free(h->du[1]); dev_free(h->dv[0]); dev_free(h->dv[1]);
    dev_free(h->Ix); dev_free(h->Iy); dev_free(h->Iz);
    dev_free(h->hin0); dev_free(h->hin1);
    if (h->stream) (void)hipStreamDestroy(h->stream);
    delete h;
}

// The launch shape of a level: the caller's, or the cheapest of 64x32 and
// 64x48 tiles with 1..14 sweeps per launch.  A sweep is its chain, barrier and
// 26 VALU instructions per pixel of the tile, halo included (VALU busy a third
// of the time at 640x480); a launch adds its ramp and, per round of 256
// workgroups, the loads and stores; deep blocks amortise those, small halos save
// work, and the grid quantises to rounds of the 256 CUs.  The model (us): 1.5 per launch, per
// round 1.5 + 0.010 per tile row and sweep.  Over 79x44 .. 1920x1080 it
// picks within 8% of the fastest of 46 measured shapes (64x64 and 8-wave
// tiles among them), e.g. 120 sweeps (us; 64x32 tiles with 4 sweeps per
// launch in parentheses): 79x44 83 (152), 638x359 127 (185), 640x480 151
// (190), 1277x719 282 (331), 1920x1080 490 (607).
JacobiShape pick_shape(const of_hs* h, int w, int hh, int sweeps)
{
    if (h->K) return JacobiShape{h->K, h->R, kHsWaves};
    JacobiShape best{4, 2, 16};
    double best_us = 0.0;
    for (int R = 2; R <= 3; R++)
        for (int K = 1; K <= 14 && K <= std::max(sweeps, 1); K++) {
            const int rows = 16 * R;
            const double launches = (sweeps + K - 1) / K;
            const double rounds = cdiv((size_t)cdiv(w, 64 - 2 * K) * cdiv(hh, rows - 2 * K), 256);
            const double us = launches * (1.5 + 1.5 * rounds) + 0.010 * rows * rounds * sweeps;
            if (best_us == 0.0 || us < best_us) {
                best_us = us;
                best = JacobiShape{K, R, 16};
            }
        }
    return best;
}

// ComputeFlow, src/hs/cuda/flow.cu:112-208, from device frames (stride s).
int hs_solve(of_hs* h, const float* dI0, const float* dI1, int width, int height, int stride,
             float alpha, int nLevels, int nWarpIters, int nSolverIters, float* du_out,
             float* dv_out, hipStream_t st)
{
    if (width != h->W || height != h->H || stride != h->stride || nLevels != h->nLevels)
        return OF_ERR_ARG;
    if (nWarpIters < 0 || nSolverIters < 0) return OF_ERR_ARG;
    const size_t fsize = (size_t)stride * height;
    int L = nLevels - 1;
    const unsigned blocks = std::min(cdiv(fsize, 256), 2048u);
    // the initial flow is read at the coarsest level, the padding columns of
    // the result are those of the finest
    hipLaunchKernelGGL(k_hs_copy2, dim3(blocks), dim3(256), 0, st, dI0, h->pI0[L], dI1, h->pI1[L], fsize,
                       h->u, h->v, std::max(fsize, (size_t)h->pS[0] * h->pH[0]));
    HS_CHECK("k_hs_copy2");
    for (; L > 0; --L) {
        hipLaunchKernelGGL(k_hs_downscale, grid2d(h->pW[L - 1], h->pH[L - 1]), dim3(256), 0, st,
                           h->pI0[L], h->pS[L], h->pI0[L - 1], h->pW[L - 1], h->pH[L - 1], h->pS[L - 1]);
        HS_CHECK("k_hs_downscale");
        hipLaunchKernelGGL(k_hs_downscale, grid2d(h->pW[L - 1], h->pH[L - 1]), dim3(256), 0, st,
                           h->pI1[L], h->pS[L], h->pI1[L - 1], h->pW[L - 1], h->pH[L - 1], h->pS[L - 1]);
        HS_CHECK("k_hs_downscale");
    }
    for (L = 0; L < nLevels; ++L) {
        const int w = h->pW[L], hh = h->pH[L], s = h->pS[L];
        for (int wi = 0; wi < nWarpIters; ++wi) {
            hipLaunchKernelGGL(k_hs_warp_derivs, dim3(cdiv(w, kWdX), cdiv(hh, kWdY)), dim3(256), 0, st,
                               h->pI0[L], h->pI1[L], w, hh, s, h->u, h->v, h->Ix, h->Iy, h->Iz,
                               (float*)nullptr);
            HS_CHECK("k_hs_warp_derivs");
            int res = 0;
            JacobiArgs a{};
            a.Ix = h->Ix;
            a.Iy = h->Iy;
            a.Iz = h->Iz;
            a.w = w;
            a.h = hh;
            a.s = s;
            a.alpha = alpha;
            OF_TRY(run_jacobi(pick_shape(h, w, hh, nSolverIters), a, h->du, h->dv, nSolverIters, true,
                              h->u, h->v, &res, st));
        }
        if (L != nLevels - 1) {
            const float scaleX = (float)h->pW[L + 1] / (float)h->pW[L];
            const float scaleY = (float)h->pH[L + 1] / (float)h->pH[L];
            hipLaunchKernelGGL(k_hs_upscale, grid2d(h->pW[L + 1], h->pH[L + 1]), dim3(256), 0, st,
                               h->u, w, hh, s, h->nu, h->pW[L + 1], h->pH[L + 1], h->pS[L + 1], scaleX);
            HS_CHECK("k_hs_upscale");
            hipLaunchKernelGGL(k_hs_upscale, grid2d(h->pW[L + 1], h->pH[L + 1]), dim3(256), 0, st,
                               h->v, w, hh, s, h->nv, h->pW[L + 1], h->pH[L + 1], h->pS[L + 1], scaleY);
            HS_CHECK("k_hs_upscale");
            float* t = h->u; h->u = h->nu; h->nu = t;
            t = h->v; h->v = h->nv; h->nv = t;
        }
    }
    // the result is in h->u/h->v, which the level loop swaps with nu/nv
    if (du_out && dv_out) {
        hipLaunchKernelGGL(k_hs_copy2, dim3(blocks), dim3(256), 0, st, h->u, du_out, h->v, dv_out, fsize,
                           (float*)nullptr, (float*)nullptr, (size_t)0);
        HS_CHECK("k_hs_copy2");
    }
    OF_HIP(hipStreamSynchronize(st));
    return OF_OK;
}

}  // namespace

extern "C" {

int of_hs_create(int nLevels, int stride, int width, int height, of_hs** out)
{
    if (!out) return OF_ERR_ARG;
    *out = nullptr;
    if (nLevels < 1 || nLevels > 32 || width < 1 || height < 1 || stride < width) return OF_ERR_ARG;
    if ((long long)stride * height >= (1ll << 31)) return OF_ERR_ARG;
    of_hs* h = new (std::nothrow) of_hs();
    if (!h) return OF_ERR_ALLOC;
    h->nLevels = nLevels;
    h->stride = stride;
    h->W = width;
    h->H = height;
    const int top = nLevels - 1;
    h->pW[top] = width; h->pH[top] = height; h->pS[top] = stride;
    for (int L = top; L > 0; --L) {
        h->pW[L - 1] = h->pW[L] / 2;
        h->pH[L - 1] = h->pH[L] / 2;
        h->pS[L - 1] = ((h->pW[L - 1] + 31) / 32) * 32;   // iAlignUp, common.cuh:47-55
        if (h->pW[L - 1] < 1 || h->pH[L - 1] < 1) { delete h; return OF_ERR_ARG; }
    }
    if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) {
        h->stream = nullptr;
        hs_release(h);
        return OF_ERR_HIP;
    }
    h->pI0 = new (std::nothrow) float*[nLevels]();
    h->pI1 = new (std::nothrow) float*[nLevels]();
    if (!h->pI0 || !h->pI1) { hs_release(h); return OF_ERR_ALLOC; }
    const size_t fsize = (size_t)stride * height;
    // coarse levels have pitches of whole 32 columns: on frames narrower than
    // 16 columns their planes are larger than the finest one's
    for (int L = 0; L < nLevels; L++) h->plane = std::max(h->plane, (size_t)h->pS[L] * h->pH[L]);
    int st = OF_OK;
    for (int L = 0; L < nLevels && !st; L++) {
        const size_t n = (size_t)h->pS[L] * h->pH[L];
        st = dev_alloc(&h->pI0[L], n);
        if (!st) st = dev_alloc(&h->pI1[L], n);
    }
    float** bufs[] = {&h->u, &h->v, &h->nu, &h->nv, &h->du[0], &h->du[1], &h->dv[0], &h->dv[1],
                      &h->Ix, &h->Iy, &h->Iz};
    float** staging[] = {&h->hin0, &h->hin1};
    for (float** b : bufs)
        if (!st) st = dev_alloc(b, h->plane);
    for (float** b : staging)
        if (!st) st = dev_alloc(b, fsize);
    if (st) { hs_release(h); return st; }
    // padding columns of strided buffers are never read by the kernels;
    // clear everything once so downloads are deterministic
    for (float** b : bufs)
        if (hipMemsetAsync(*b, 0, h->plane * sizeof(float), h->stream) != hipSuccess) st = OF_ERR_HIP;
    for (float** b : staging)
        if (hipMemsetAsync(*b, 0, fsize * sizeof(float), h->stream) != hipSuccess) st = OF_ERR_HIP;
    for (int L = 0; L < nLevels; L++) {
        const size_t n = (size_t)h->pS[L] * h->pH[L];
        if (hipMemsetAsync(h->pI0[L], 0, n * sizeof(float), h->stream) != hipSuccess) st = OF_ERR_HIP;
        if (hipMemsetAsync(h->pI1[L], 0, n * sizeof(float), h->stream) != hipSuccess) st = OF_ERR_HIP;
    }
    if (!st && hipStreamSynchronize(h->stream) != hipSuccess) st = OF_ERR_HIP;
    if (st) { hs_release(h); return st; }
    *out = h;
    return OF_OK;
}

void of_hs_destroy(of_hs* h) { hs_release(h); }

int of_hs_set_jacobi_shape(of_hs* h, int sweeps_per_launch, int rows_per_wave)
{
    if (!h) return OF_ERR_ARG;
    if (!jacobi_shape_ok(sweeps_per_launch, rows_per_wave)) return OF_ERR_UNSUPPORTED;
    h->K = sweeps_per_launch;
    h->R = rows_per_wave;
    return OF_OK;
}

int of_hs_compute_device(of_hs* h, const float* dI0, const float* dI1, int width, int height,
                         int stride, float alpha, int nLevels, int nWarpIters, int nSolverIters,
                         float* du, float* dv, void* stream)
{
    if (!h || !dI0 || !dI1 || !du || !dv) return OF_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;   // NULL: the HIP null stream
    return hs_solve(h, dI0, dI1, width, height, stride, alpha, nLevels, nWarpIters, nSolverIters,
                    du, dv, st);
}

int of_hs_compute(of_hs* h, const float* I0, const float* I1, int width, int height, int stride,
                  float alpha, int nLevels, int nWarpIters, int nSolverIters, float* u, float* v)
{
    if (!h || !I0 || !I1 || !u || !v) return OF_ERR_ARG;
    if (width != h->W || height != h->H || stride != h->stride) return OF_ERR_ARG;
    const size_t fsize = (size_t)stride * height;
    OF_HIP(hipMemcpyAsync(h->hin0, I0, fsize * sizeof(float), hipMemcpyHostToDevice, h->stream));
    OF_HIP(hipMemcpyAsync(h->hin1, I1, fsize * sizeof(float), hipMemcpyHostToDevice, h->stream));
    OF_TRY(hs_solve(h, h->hin0, h->hin1, width, height, stride, alpha, nLevels, nWarpIters,
                    nSolverIters, nullptr, nullptr, h->stream));
    // read the buffers after the solve: every level but the last swaps u
    // with nu (and v with nv), so which one holds the flow depends on the
    // level count
    OF_HIP(hipMemcpyAsync(u, h->u, fsize * sizeof(float), hipMemcpyDeviceToHost, h->stream));
    OF_HIP(hipMemcpyAsync(v, h->v, fsize * sizeof(float), hipMemcpyDeviceToHost, h->stream));
    OF_HIP(hipStreamSynchronize(h->stream));
    return OF_OK;
}

// ---- per-kernel test entry points (amdflow_debug.h) ----

int of_dbg_hs_jacobi(const float* du, const float* dv, const float* Ix, const float* Iy,
                     const float* Iz, int w, int h, float alpha, int iters, int K, int R,
                     float* du_out, float* dv_out)
{
    if (!du || !dv || !Ix || !Iy || !Iz || !du_out || !dv_out || w < 1 || h < 1 || iters < 0)
        return OF_ERR_ARG;
    if (!jacobi_shape_ok(K, R)) return OF_ERR_UNSUPPORTED;
    const size_t n = (size_t)w * h;
    float* b[7] = {};
    int st = OF_OK;
    for (float*& p : b)
        if (!st) st = dev_alloc(&p, n);
    if (!st) {
        const float* src[5] = {du, dv, Ix, Iy, Iz};
        for (int i = 0; i < 5 && !st; i++)
            if (hipMemcpy(b[i], src[i], n * sizeof(float), hipMemcpyHostToDevice) != hipSuccess)
                st = OF_ERR_HIP;
    }
    int res = 0;
    float* dus[2] = {b[0], b[5]};
    float* dvs[2] = {b[1], b[6]};
    JacobiArgs a{};
    a.Ix = b[2];
    a.Iy = b[3];
    a.Iz = b[4];
    a.w = w;
    a.h = h;
    a.s = w;
    a.alpha = alpha;
    if (!st) st = run_jacobi(JacobiShape{K, R, kHsWaves}, a, dus, dvs, iters, false, nullptr, nullptr, &res, nullptr);
    if (!st && hipMemcpy(du_out, dus[res], n * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) st = OF_ERR_HIP;
    if (!st && hipMemcpy(dv_out, dvs[res], n * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) st = OF_ERR_HIP;
    for (float*& p : b) dev_free(p);
    return st;
}

int of_dbg_hs_warp_derivatives(const float* I0, const float* I1, const float* u, const float* v,
                               int w, int h, float* I1w, float* Ix, float* Iy, float* Iz)
{
    if (!I0 || !I1 || !u || !v || !I1w || !Ix || !Iy || !Iz || w < 1 || h < 1) return OF_ERR_ARG;
    const size_t n = (size_t)w * h;
    float* b[8] = {};
    int st = OF_OK;
    for (float*& p : b)
        if (!st) st = dev_alloc(&p, n);
    const float* src[4] = {I0, I1, u, v};
    for (int i = 0; i < 4 && !st; i++)
        if (hipMemcpy(b[i], src[i], n * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) st = OF_ERR_HIP;
    if (!st) {
        hipLaunchKernelGGL(k_hs_warp_derivs, dim3(cdiv(w, kWdX), cdiv(h, kWdY)), dim3(256), 0, nullptr, b[0],
                           b[1], w, h, w, b[2], b[3], b[5], b[6], b[7], b[4]);
        if (hipGetLastError() != hipSuccess) st = OF_ERR_HIP;
    }
    float* dst[4] = {I1w, Ix, Iy, Iz};
    for (int i = 0; i < 4 && !st; i++)
        if (hipMemcpy(dst[i], b[4 + i], n * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) st = OF_ERR_HIP;
    for (float*& p : b) dev_free(p);
    return st;
}

// Runs one pyramid step (down: 2x2 box; up: x2 flow upscale times `scale`)
// on a dense w x h plane into a dense nw x nh plane.
static int dbg_hs_resample(const float* src, int w, int h, float* out, int nw, int nh, bool up,
                           float scale)
{
    if (!src || !out || w < 1 || h < 1 || nw < 1 || nh < 1) return OF_ERR_ARG;
    // the box reads rows/columns 2i and 2i+1 of the source
    if (!up && (2 * (long long)nw > w || 2 * (long long)nh > h)) return OF_ERR_ARG;
    const size_t n = (size_t)w * h, nn = (size_t)nw * nh;
    float *ds = nullptr, *dd = nullptr;
    int st = dev_alloc(&ds, n);
    if (!st) st = dev_alloc(&dd, nn);
    if (!st && hipMemcpy(ds, src, n * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) st = OF_ERR_HIP;
    if (!st) {
        if (up)
            hipLaunchKernelGGL(k_hs_upscale, grid2d(nw, nh), dim3(256), 0, nullptr, ds, w, h, w, dd,
                               nw, nh, nw, scale);
        else
            hipLaunchKernelGGL(k_hs_downscale, grid2d(nw, nh), dim3(256), 0, nullptr, ds, w, dd, nw,
                               nh, nw);
        if (hipGetLastError() != hipSuccess) st = OF_ERR_HIP;
    }
    if (!st && hipMemcpy(out, dd, nn * sizeof(float), hipMemcpyDeviceToHost) != hipSuccess) st = OF_ERR_HIP;
    dev_free(ds);
    dev_free(dd);
    return st;
}

int of_dbg_hs_downscale(const float* src, int w, int h, float* out, int nw, int nh)
{
    return dbg_hs_resample(src, w, h, out, nw, nh, false, 1.0f);
}

int of_dbg_hs_upscale(const float* src, int w, int h, float* out, int nw, int nh, float scale)
{
    return dbg_hs_resample(src, w, h, out, nw, nh, true, scale);
}

}  // extern "C"
