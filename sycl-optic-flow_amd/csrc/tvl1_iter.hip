// tvl1_iter.hip -- the TV-L1 primal-dual iterations (tvl1.cpp:214-292).
//
// Drivers of the tile cores:
//   k_tvl1_iter<K,R>         one launch = K iterations; the last workgroup to
//                            finish evaluates the stopping rule; the host keeps
//                            a few launches queued;
//   k_tvl1_persist<K,R>      one launch of a co-resident grid = a whole
//                            warping; chunks of K iterations separated by a
//                            grid barrier, every workgroup evaluating the
//                            stopping rule on the same data;
//   k_tvl1_persist_nbr<K,R>  the same without grid barriers: tiles wait for
//                            their neighbours' flags, a referee workgroup
//                            decides;
//   k_tvl1_persist_tag<T,K>  square tiles with a CU each, state in registers,
//                            tagged values in place of flags;
//   k_tvl1_single<K>         scales of at most 32 x 32 in one workgroup;
//   k_ls_iter<K,R>           one launch = K iterations of many pairs.
// Arithmetic follows the reference operation by operation; the library is
// built with -ffp-contract=off.
#include <algorithm>
#include <atomic>
#include <cstdlib>

#include "device_math.hpp"
#include "lockstep.hpp"
#include "tvl1_kernels.hpp"

namespace amdflow {

// Divergence at one pixel from the current value and the left/up neighbours
// with the border rules of mask.cpp:31-77.  Written with selects; every
// candidate is the exact expression of its reference case (the first/last
// column cases associate left to right as written at :81-82).
__device__ __forceinline__ float div_rule(float v1, float v1l, float v2, float v2u, bool fr,
                                          bool lr, bool fc, bool lc)
{
    const float a = fc ? v1 : (lc ? -v1l : (v1 - v1l));
    const float t_first_row = a + v2;               // :70, corners :86-87
    const float t_last_row = a - v2u;               // :71, corners :88-89
    const float t_edge_col = (a + v2) - v2u;        // :81-82
    const float t_body = a + (v2 - v2u);            // :59
    return fr ? t_first_row : (lr ? t_last_row : ((fc || lc) ? t_edge_col : t_body));
}

// Thresholding operator TH, tvl1.cpp:221-245, branch-free: the three
// reference cases multiply the warped gradient by l_t, -l_t or -rho/grad,
// and the `grad < 1e-10` case stores +0 exactly as the reference does.
__device__ __forceinline__ void th_step(float rc, float gx, float gy, float u1, float u2,
                                        float l_t, float& v1, float& v2)
{
    const float grad = (gx * gx) + (gy * gy);
    const float rho = rc + ((gx * u1) + (gy * u2));
    const float fi = -rho / grad;
    const float lg = l_t * grad;   // (-l_t) * grad is -lg bit for bit
    const bool c1 = rho >= -lg;
    const bool c2 = rho > lg;
    const bool c3 = grad < 1E-10f;
    const bool zero = c1 && !c2 && c3;
    const float k = c1 ? (c2 ? -l_t : fi) : l_t;
    const float d1 = zero ? 0.0f : k * gx;
    const float d2 = zero ? 0.0f : k * gy;
    v1 = u1 + d1;
    v2 = u2 + d2;
}

// g = 1 + taut*hypot(fx, fy) and 1/g in double, both for one component of
// the dual update.
struct DualDiv {
    float g;
    double r;
    unsigned near;   // below 2^12: the root is too close to a float rounding boundary to be sure
};

__device__ __forceinline__ DualDiv dual_div(float fx, float fy, float taut)
{
    DualDiv d;
    const double x = (double)fx, y = (double)fy;
    // the squares are exact in double.  The added 2^-200 keeps a zero gradient
    // off the root's pole and otherwise only reaches sums below 2^-140, whose
    // root leaves g at 1 (taut < 2^40).
    const double s = __builtin_fma(x, x, __builtin_fma(y, y, 0x1p-200));
    const double q = __builtin_amdgcn_rsq(s);
    const double h0 = s * q;
    const double h = __builtin_fma(0.5 * h0, __builtin_fma(-h0, q, 1.0), h0);
    // h is within 2^-47 of sqrt(s) (the hardware root seed is within 2^-24).
    // Its float rounding is that of the exact double root unless the 29
    // dropped bits are within 2^8 of half a float ulp (2^28): 2^11 of 2^31
    // after the shift.
    d.near = ((unsigned)__double2loint(h) << 3) + (0x80000000u + (1u << 11));
    d.g = 1.0f + taut * (float)h;
    // 1/g to about an ulp: the float reciprocal and one cubic step
    const double g = (double)d.g, r0 = (double)__builtin_amdgcn_rcpf(d.g);
    const double e = __builtin_fma(-g, r0, 1.0);
    d.r = __builtin_fma(__builtin_fma(e, e, e), r0, r0);
    return d;
}

// The dual update of one pixel: p = (p + taut*grad u)/(1 + taut*|grad u|)
// for both components (cblas_saxpy, then the division, tvl1.cpp:280-291).
// The kernels are bound by VALU issue and this is the larger half of an
// iteration, so it runs without the IEEE sequences (per pixel 2 roots of 21
// instructions' cost and 4 divisions of 10): the root is refined once and
// rounded, the quotients are products with a shared double reciprocal.  A
// float quotient is never within 2^-49 of a rounding boundary and the product
// is within 2^-52 of it, so the bits are the division's; a subnormal quotient
// can lie on a boundary only if g is an even integer, and for 2 and 4 the
// reciprocal is exact.  Roots near a boundary, g >= 6, infinities and NaN take
// the full sequences, for the whole wave (the roots of about one row in 8000).
__device__ __forceinline__ void dual_step(float fx1, float fy1, float fx2, float fy2, float taut,
                                          float& p11, float& p12, float& p21, float& p22)
{
    const float n11 = p11 + taut * fx1, n12 = p12 + taut * fy1;
    const float n21 = p21 + taut * fx2, n22 = p22 + taut * fy2;
    const DualDiv a = dual_div(fx1, fy1, taut), b = dual_div(fx2, fy2, taut);
    const bool sure = (a.g < 6.0f) & (b.g < 6.0f) & (min(a.near, b.near) >= (1u << 12)) & (taut < 0x1p40f);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(!sure) == 0ull, 1)) {
        p11 = (float)((double)n11 * a.r);
        p12 = (float)((double)n12 * a.r);
        p21 = (float)((double)n21 * b.r);
        p22 = (float)((double)n22 * b.r);
    } else {
        const float g1 = 1.0f + taut * hypot_fin(fx1, fy1);
        const float g2 = 1.0f + taut * hypot_fin(fx2, fy2);
        p11 = n11 / g1;
        p12 = n12 / g1;
        p21 = n21 / g2;
        p22 = n22 / g2;
    }
}

// v plus the value of the lane that the DPP control names (0 where there is
// none or the row mask excludes the lane).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add_f64(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, true);
    const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, true);
    return v + __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// Sum over the wave, valid in lane 63: rows of 16 by shifts, then the rows'
// totals broadcast.  DPP moves instead of cross-lane LDS permutes: the sums of
// a tile's errors run once per tile and chunk (1920x1080, 2 iterations per
// chunk: a seventh of a tile's instructions before).
__device__ __forceinline__ double wave_sum_f64(double v)
{
    v = dpp_add_f64<0x111, 0xf>(v);   // row_shr:1
    v = dpp_add_f64<0x112, 0xf>(v);   // row_shr:2
    v = dpp_add_f64<0x114, 0xf>(v);   // row_shr:4
    v = dpp_add_f64<0x118, 0xf>(v);   // row_shr:8
    v = dpp_add_f64<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
    return dpp_add_f64<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
}

// A value that every lane holds alike, in a scalar register: what depends on
// it (buffer pointers, tile addresses, loop exits) stays scalar too.
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Widest frame whose tile rows are addressed by 32-bit lane offsets (8 rows
// of 4-byte values stay below 2^32 bytes).
constexpr int kMaxLaneCols = 1 << 26;

// A plane at an element offset, kept in scalar registers: accesses relative to
// it take a 32-bit lane offset.  (Otherwise the compiler adds the lane to each
// plane's base ahead of the loops, in vector registers, and the offset with
// 64-bit vector instructions per access.)
struct PlanePtr {
    typedef __attribute__((address_space(1))) char gchar;
    typedef __attribute__((address_space(1))) float gfloat;
    gchar* p;
    __device__ __forceinline__ PlanePtr(const float* plane, ptrdiff_t o) : p((gchar*)(plane + o))
    {
        asm("" : "+s"(p));
    }
    __device__ __forceinline__ gfloat* at(unsigned bytes) const { return (gfloat*)(p + bytes); }
};

// Loads and stores of the iteration state.  COH: device-scope atomic
// accesses, coherent across XCDs without cache maintenance (used when other
// workgroups of the same launch read the values).
template <bool COH, class P>
__device__ __forceinline__ float ld(const P* p)
{
    if constexpr (COH) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else return *p;
}

template <bool COH, class P>
__device__ __forceinline__ void st(P* p, float v)
{
    if constexpr (COH) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}

// Called by every thread of a tile's workgroup.  ready(): before the loads of
// the state (the warping's constants are on their way by then); store():
// between the iterations and the stores.  false ends the tile there (the
// neighbour-synchronised warping waits for its neighbours and checks its
// speculative chunk in them).  The default does neither.
struct NoSync {
    __device__ bool ready() const { return true; }
    __device__ bool store() const { return true; }
};

// One LDS row per wave and exchanged quantity; NW waves per workgroup.
template <int NW>
struct TileSharedN {
    float a[NW][64], b[NW][64], c[NW][64], d[NW][64];
};
using TileShared = TileSharedN<4>;

// kk (<= K) iterations on tile (bx, by): reads buffer `cur`, writes the
// central tile into buffer cur^1, adds each iteration's per-lane error sum
// over the central tile to acc[t].
//
// One workgroup = NW waves; the extended tile is 64 columns (one per lane) by
// NW*R rows (R consecutive rows per wave, in registers).  Horizontal
// neighbours come from DPP lane shifts, vertical ones from the lane's own
// registers or, across waves, from one LDS row.  Values within K pixels of
// the tile edge go stale one pixel per iteration; the central (64-2K) x
// (NW*R-2K) pixels are exact.
template <int K, int R, bool COH, bool INNER, int NW, class Sync>
__device__ __forceinline__ void tile_iterate_impl(const IterArgs& a, int bx, int by, int cur, int kk,
                                                  double (&acc)[K], TileSharedN<NW>& sh, Sync& sync)
{
    constexpr int TW = 64 - 2 * K;
    constexpr int TH = NW * R - 2 * K;
    bx = uniform(bx);
    by = uniform(by);
    cur = uniform(cur);
    const int lane = threadIdx.x & 63;
    const int wave = uniform(threadIdx.x >> 6);
    const int nx = a.nx, ny = a.ny;
    const int x = bx * TW - K + lane;
    const int ybase = by * TH - K + wave * R;
    const int oy0 = by * TH;
    // INNER: the extended tile lies within columns 1..nx-2 and rows 1..ny-2,
    // so every border test below is known and folds away, and the frame is
    // at most kMaxLaneCols wide
    const bool xin = INNER || (x >= 0 && x < nx);
    const bool xout = xin && lane >= K && lane < K + TW;
    const bool fc = !INNER && x == 0, lc = !INNER && x == nx - 1;
    // waves holding no first/last image column take the body formula of the
    // divergence on every row away from the first/last image row
    const bool edge_cols = !INNER && __any(fc || lc);

    // (selects: an indexed kernel argument would be loaded per lane)
    const float* uin = cur ? a.u[1] : a.u[0];
    const float* pin = cur ? a.p[1] : a.p[0];
    const size_t plane = (size_t)a.plane;

    float u1[R], u2[R], p11[R], p12[R], p21[R], p22[R], gx[R], gy[R], rc[R];
    const ptrdiff_t o0 = (ptrdiff_t)ybase * nx + (bx * TW - K);   // the wave's first pixel
    const unsigned ob = (unsigned)lane * 4u, onx = (unsigned)nx * 4u;
    if constexpr (INNER) {
        const PlanePtr GX(a.wx, o0), GY(a.wy, o0), RC(a.rhoc, o0);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const unsigned o = ob + (unsigned)r * onx;
            gx[r] = *GX.at(o);
            gy[r] = *GY.at(o);
            rc[r] = *RC.at(o);
        }
        if (!sync.ready()) return;
        const PlanePtr U1(uin, o0), U2(uin + plane, o0), P11(pin, o0), P12(pin + plane, o0),
            P21(pin + 2 * plane, o0), P22(pin + 3 * plane, o0);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const unsigned o = ob + (unsigned)r * onx;
            u1[r] = ld<COH>(U1.at(o));
            u2[r] = ld<COH>(U2.at(o));
            p11[r] = ld<COH>(P11.at(o));
            p12[r] = ld<COH>(P12.at(o));
            p21[r] = ld<COH>(P21.at(o));
            p22[r] = ld<COH>(P22.at(o));
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int y = ybase + r;
            gx[r] = gy[r] = rc[r] = 0.0f;
            if (xin && y >= 0 && y < ny) {
                const size_t idx = (size_t)y * nx + x;
                gx[r] = a.wx[idx];
                gy[r] = a.wy[idx];
                rc[r] = a.rhoc[idx];
            }
        }
        if (!sync.ready()) return;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int y = ybase + r;
            u1[r] = u2[r] = p11[r] = p12[r] = p21[r] = p22[r] = 0.0f;
            if (xin && y >= 0 && y < ny) {
                const size_t idx = (size_t)y * nx + x;
                u1[r] = ld<COH>(uin + idx);
                u2[r] = ld<COH>(uin + plane + idx);
                p11[r] = ld<COH>(pin + idx);
                p12[r] = ld<COH>(pin + plane + idx);
                p21[r] = ld<COH>(pin + 2 * plane + idx);
                p22[r] = ld<COH>(pin + 3 * plane + idx);
            }
        }
    }

    const float l_t = a.l_t, theta = a.theta, taut = a.taut;
#pragma unroll
    for (int t = 0; t < K; t++) {
        if (t < kk) {
            // ---- u update: TH, divergence of p, u = v + theta*div p ----
            sh.a[wave][lane] = p12[R - 1];
            sh.b[wave][lane] = p22[R - 1];
            __syncthreads();
            const float up12 = wave ? sh.a[wave - 1][lane] : p12[0];
            const float up22 = wave ? sh.b[wave - 1][lane] : p22[0];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int y = ybase + r;
                const float p11l = lane_left(p11[r]);
                const float p21l = lane_left(p21[r]);
                const float p12u = r ? p12[r - 1] : up12;
                const float p22u = r ? p22[r - 1] : up22;
                const bool fr = !INNER && y == 0, lr = !INNER && y == ny - 1;
                float div1, div2;
                if (!edge_cols && !fr && !lr) {   // uniform branch: interior rows of interior waves
                    div1 = (p11[r] - p11l) + (p12[r] - p12u);
                    div2 = (p21[r] - p21l) + (p22[r] - p22u);
                } else {
                    div1 = div_rule(p11[r], p11l, p12[r], p12u, fr, lr, fc, lc);
                    div2 = div_rule(p21[r], p21l, p22[r], p22u, fr, lr, fc, lc);
                }
                float v1, v2;
                th_step(rc[r], gx[r], gy[r], u1[r], u2[r], l_t, v1, v2);
                const float nu1 = v1 + theta * div1;
                const float nu2 = v2 + theta * div2;
                const float e1 = nu1 - u1[r], e2 = nu2 - u2[r];
                const float e = e1 * e1 + e2 * e2;
                const bool mine = xout && y >= oy0 && y < oy0 + TH && (INNER || y < ny);
                acc[t] += (double)(mine ? e : 0.0f);
                u1[r] = nu1;
                u2[r] = nu2;
            }
            // ---- p update: forward gradient of u, g, p = (p + taut*grad)/g ----
            sh.c[wave][lane] = u1[0];
            sh.d[wave][lane] = u2[0];
            __syncthreads();
            const float dn1 = wave < NW - 1 ? sh.c[wave + 1][lane] : u1[R - 1];
            const float dn2 = wave < NW - 1 ? sh.d[wave + 1][lane] : u2[R - 1];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int y = ybase + r;
                const float u1r = lane_right(u1[r]);
                const float u2r = lane_right(u2[r]);
                const float u1d = r < R - 1 ? u1[r + 1] : dn1;
                const float u2d = r < R - 1 ? u2[r + 1] : dn2;
                const bool xl = INNER || x < nx - 1, yl = INNER || y < ny - 1;
                const float fx1 = xl ? u1r - u1[r] : 0.0f;
                const float fy1 = yl ? u1d - u1[r] : 0.0f;
                const float fx2 = xl ? u2r - u2[r] : 0.0f;
                const float fy2 = yl ? u2d - u2[r] : 0.0f;
                dual_step(fx1, fy1, fx2, fy2, taut, p11[r], p12[r], p21[r], p22[r]);
            }
        }
    }

    if (!sync.store()) return;
    float* uout = cur ? a.u[0] : a.u[1];
    float* pout = cur ? a.p[0] : a.p[1];
    if (!xout) return;
    if constexpr (INNER) {
        const PlanePtr U1(uout, o0), U2(uout + plane, o0), P11(pout, o0), P12(pout + plane, o0),
            P21(pout + 2 * plane, o0), P22(pout + 3 * plane, o0);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int y = ybase + r;
            if (y >= oy0 && y < oy0 + TH) {
                const unsigned o = ob + (unsigned)r * onx;
                st<COH>(U1.at(o), u1[r]);
                st<COH>(U2.at(o), u2[r]);
                st<COH>(P11.at(o), p11[r]);
                st<COH>(P12.at(o), p12[r]);
                st<COH>(P21.at(o), p21[r]);
                st<COH>(P22.at(o), p22[r]);
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int y = ybase + r;
            if (y >= oy0 && y < oy0 + TH && y < ny) {
                const size_t idx = (size_t)y * nx + x;
                st<COH>(uout + idx, u1[r]);
                st<COH>(uout + plane + idx, u2[r]);
                st<COH>(pout + idx, p11[r]);
                st<COH>(pout + plane + idx, p12[r]);
                st<COH>(pout + 2 * plane + idx, p21[r]);
                st<COH>(pout + 3 * plane + idx, p22[r]);
            }
        }
    }
}

// Tiles whose extended area (64 columns x 4R rows from (bx*TW-K, by*TH-K))
// stays clear of the image border run the INNER variant.
template <int K, int R, bool COH, int NW, class Sync>
__device__ __forceinline__ void tile_iterate(const IterArgs& a, int bx, int by, int cur, int kk,
                                             double (&acc)[K], TileSharedN<NW>& sh, Sync& sync)
{
    constexpr int TW = 64 - 2 * K;
    constexpr int TH = NW * R - 2 * K;
    const int x0 = bx * TW - K, y0 = by * TH - K;
    const bool inner = x0 >= 1 && x0 + 63 <= a.nx - 2 && y0 >= 1 && y0 + NW * R - 1 <= a.ny - 2 &&
                       a.nx <= kMaxLaneCols;
    if (inner) tile_iterate_impl<K, R, COH, true, NW>(a, bx, by, cur, kk, acc, sh, sync);
    else tile_iterate_impl<K, R, COH, false, NW>(a, bx, by, cur, kk, acc, sh, sync);
}

// Square tiles for the small scales: one workgroup of T*T lanes covers a
// T x T pixel tile, one pixel per lane, neighbours exchanged through LDS.
// With K iterations per launch the central (T-2K) x (T-2K) pixels are
// exact.  One pixel per lane and more workgroups hide less latency per
// lane but keep many more CUs busy than 64-column tiles at scales of a few
// ten thousand pixels (120x68: 1.2 instead of 3.3 us per iteration).  All
// neighbours go through LDS: at T = 32, where a wave is two whole rows, lane
// shifts for the horizontal ones cost more than they saved (641x479, two tiles
// per CU: 0.48 against 0.44 ms).
constexpr int kSqTile = 16;   // the tile of launch shapes with rows_per_wave 0

// p exchange in a..d, u exchange in e, f: the two halves of an iteration
// use different arrays, so each needs one barrier, between its writes and
// its reads.  A half's next writes come after the other half's barrier,
// which every thread reaches only after its reads of this half.
template <int T>
struct SqShared {
    float a[T][T + 1], b[T][T + 1], c[T][T + 1], d[T][T + 1], e[T][T + 1], f[T][T + 1];
};

// One pixel of a square tile: its state, the warping's constants, and where
// it lies.
struct SqPixel {
    float u1, u2, p11, p12, p21, p22;
    float gx, gy, rc;
    bool fc, lc, fr, lr;   // first/last image column and row
    bool mine;             // its error counts
};

// kk (<= K) iterations of a tile of T columns (one pixel per lane, row ly =
// threadIdx.x / T of the workgroup's rows), each adding its error term to
// acc[t].  Same per-pixel expressions as tile_iterate_impl; pixels outside
// the image never feed pixels inside (the border rules do not read across
// the border).
template <int T, int K>
__device__ __forceinline__ void sq_iterations(const IterArgs& a, SqPixel& q, int kk, int rows,
                                              double (&acc)[K], SqShared<T>& sh)
{
    const int lx = threadIdx.x % T, ly = threadIdx.x / T;
    // neighbour slots, clamped to the tile: the edge lanes read their own
    // slot (their results are outside the exact centre)
    const int xm = lx > 0 ? lx - 1 : lx, xp = lx < T - 1 ? lx + 1 : lx;
    const int ym = ly > 0 ? ly - 1 : ly, yp = ly < rows - 1 ? ly + 1 : ly;
    // waves off the image border take the body formulas
    const bool edge = __any(q.fc || q.lc || q.fr || q.lr);
    const float l_t = a.l_t, theta = a.theta, taut = a.taut;
#pragma unroll
    for (int t = 0; t < K; t++) {
        if (t < kk) {
            // ---- u update: TH, divergence of p, u = v + theta*div p ----
            sh.a[ly][lx] = q.p11;
            sh.b[ly][lx] = q.p21;
            sh.c[ly][lx] = q.p12;
            sh.d[ly][lx] = q.p22;
            __syncthreads();
            const float p11l = sh.a[ly][xm], p21l = sh.b[ly][xm];
            const float p12u = sh.c[ym][lx], p22u = sh.d[ym][lx];
            float div1 = (q.p11 - p11l) + (q.p12 - p12u);
            float div2 = (q.p21 - p21l) + (q.p22 - p22u);
            if (edge) {
                div1 = div_rule(q.p11, p11l, q.p12, p12u, q.fr, q.lr, q.fc, q.lc);
                div2 = div_rule(q.p21, p21l, q.p22, p22u, q.fr, q.lr, q.fc, q.lc);
            }
            float v1, v2;
            th_step(q.rc, q.gx, q.gy, q.u1, q.u2, l_t, v1, v2);
            const float nu1 = v1 + theta * div1;
            const float nu2 = v2 + theta * div2;
            const float e1 = nu1 - q.u1, e2 = nu2 - q.u2;
            const float e = e1 * e1 + e2 * e2;
            acc[t] += (double)(q.mine ? e : 0.0f);
            q.u1 = nu1;
            q.u2 = nu2;
            // ---- p update: forward gradient of u, g, p = (p + taut*grad)/g ----
            sh.e[ly][lx] = q.u1;
            sh.f[ly][lx] = q.u2;
            __syncthreads();
            const float u1r = sh.e[ly][xp], u2r = sh.f[ly][xp];
            const float u1d = sh.e[yp][lx], u2d = sh.f[yp][lx];
            float fx1 = u1r - q.u1, fy1 = u1d - q.u1, fx2 = u2r - q.u2, fy2 = u2d - q.u2;
            if (edge) {
                fx1 = q.lc ? 0.0f : fx1;
                fy1 = q.lr ? 0.0f : fy1;
                fx2 = q.lc ? 0.0f : fx2;
                fy2 = q.lr ? 0.0f : fy2;
            }
            dual_step(fx1, fy1, fx2, fy2, taut, q.p11, q.p12, q.p21, q.p22);
        }
    }
}

__device__ __forceinline__ void sq_load_constants(const IterArgs& a, SqPixel& q, bool in, size_t idx)
{
    q.gx = q.gy = q.rc = 0.0f;
    if (in) {
        q.gx = a.wx[idx];
        q.gy = a.wy[idx];
        q.rc = a.rhoc[idx];
    }
}

template <bool COH>
__device__ __forceinline__ void sq_load_state(const IterArgs& a, SqPixel& q, bool in, size_t idx, int cur)
{
    const size_t plane = (size_t)a.plane;
    const float* uin = cur ? a.u[1] : a.u[0];
    const float* pin = cur ? a.p[1] : a.p[0];
    q.u1 = q.u2 = q.p11 = q.p12 = q.p21 = q.p22 = 0.0f;
    if (in) {
        q.u1 = ld<COH>(uin + idx);
        q.u2 = ld<COH>(uin + plane + idx);
        q.p11 = ld<COH>(pin + idx);
        q.p12 = ld<COH>(pin + plane + idx);
        q.p21 = ld<COH>(pin + 2 * plane + idx);
        q.p22 = ld<COH>(pin + 3 * plane + idx);
    }
}

template <bool COH>
__device__ __forceinline__ void sq_store_state(const IterArgs& a, const SqPixel& q, size_t idx, int cur)
{
    const size_t plane = (size_t)a.plane;
    float* uout = cur ? a.u[1] : a.u[0];
    float* pout = cur ? a.p[1] : a.p[0];
    st<COH>(uout + idx, q.u1);
    st<COH>(uout + plane + idx, q.u2);
    st<COH>(pout + idx, q.p11);
    st<COH>(pout + plane + idx, q.p12);
    st<COH>(pout + 2 * plane + idx, q.p21);
    st<COH>(pout + 3 * plane + idx, q.p22);
}

// kk (<= K) iterations on square tile (bx, by): reads buffer `cur`, writes
// the central tile into buffer cur^1, adds each iteration's per-lane error
// term over the central tile to acc[t].
template <int T, int K, bool COH, class Sync>
__device__ __forceinline__ void tile_iterate_sq(const IterArgs& a, int bx, int by, int cur, int kk,
                                                double (&acc)[K], SqShared<T>& sh, Sync& sync)
{
    constexpr int C = T - 2 * K;
    const int lx = threadIdx.x % T, ly = threadIdx.x / T;
    const int nx = a.nx, ny = a.ny;
    const int x = bx * C - K + lx, y = by * C - K + ly;
    const bool in = x >= 0 && x < nx && y >= 0 && y < ny;
    const size_t idx = (size_t)y * nx + x;
    SqPixel q;
    q.fc = x == 0;
    q.lc = x == nx - 1;
    q.fr = y == 0;
    q.lr = y == ny - 1;
    q.mine = in && lx >= K && lx < K + C && ly >= K && ly < K + C;
    sq_load_constants(a, q, in, idx);
    if (!sync.ready()) return;
    sq_load_state<COH>(a, q, in, idx, cur);
    sq_iterations<T, K>(a, q, kk, T, acc, sh);
    if (!sync.store()) return;
    if (q.mine) sq_store_state<COH>(a, q, idx, cur ^ 1);
}

// Workgroup sum of the per-lane partials, fixed order: wave tree, then
// waves 0..NW-1 left to right.  Result valid in thread t for t < K (thread t
// holds sum t).
template <int K, int NW = 4>
__device__ __forceinline__ double block_sum(const double (&acc)[K], double (*sh_err)[K], int t_out)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int t = 0; t < K; t++) {
        const double v = wave_sum_f64(acc[t]);
        if (lane == 63) sh_err[wave][t] = v;
    }
    __syncthreads();
    double s = 0.0;
    if (t_out < K) {
        s = sh_err[0][t_out];
#pragma unroll
        for (int w = 1; w < NW; w++) s += sh_err[w][t_out];
    }
    __syncthreads();
    return s;
}

// Sums over all workgroups of columns t < kk of `part` (column t holds nb
// entries at part + t*nb), fixed order per column: thread j sums entries j,
// j+64*NW, ...; then wave trees and waves 0..NW-1 left to right.  All
// columns are read in one pass, so the sums cost one memory round trip.
// Identical in every workgroup that calls it on the same data; out[t] is
// valid in every thread after the call (sh: K*NW doubles of LDS).
template <int K, int NW>
__device__ __forceinline__ void grid_sums(const double* part, unsigned nb, int kk, double* sh,
                                          double* out)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double s[K];
#pragma unroll
    for (int t = 0; t < K; t++) s[t] = 0.0;
    for (unsigned j = threadIdx.x; j < nb; j += 64 * NW) {
#pragma unroll
        for (int t = 0; t < K; t++)
            if (t < kk)
                s[t] += __hip_atomic_load(part + (size_t)t * nb + j, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int t = 0; t < K; t++) {
        const double v = wave_sum_f64(s[t]);
        if (lane == 63) sh[t * NW + wave] = v;
    }
    __syncthreads();
    if (threadIdx.x < (unsigned)K) {
        double tot = sh[threadIdx.x * NW];
#pragma unroll
        for (int w = 1; w < NW; w++) tot += sh[threadIdx.x * NW + w];
        out[threadIdx.x] = tot;
    }
    __syncthreads();
}

// The stopping rule applied to kk error sums after iteration n0 (1-based
// iterations n0+1 .. n0+kk): returns the number of iterations to keep when
// the warping stops inside or at the end of this chunk, 0 to continue.
// tvl1.cpp:214-216: continue while error > epsilon^2 and n < max.
__device__ __forceinline__ int stop_after(const double* tot, int kk, int n0, const IterArgs& a)
{
    for (int t = 0; t < kk; t++) {
        const double err = tot[t] / (double)a.plane;
        if (!(err > a.eps2)) return t + 1;
    }
    if (n0 + kk >= a.max_iter) return kk;
    return 0;
}

// Workgroups of 256 per CU the 4-wave iteration kernels are compiled for:
// 3, i.e. 3 waves per SIMD, which caps them at 168 VGPRs (allocated in steps
// of 8 out of 512).  Without the cap the largest shapes took 170 registers
// and fell to 2 waves per SIMD, and the 1920x1080 warping slowed by 10%.
constexpr int kIterBlocksPerCU = 3;

// Waves per workgroup of the one-pair iteration kernels.  A launch shape
// (K, R) names tiles of 64 x 4R pixels; they run as 8 waves of R/2 rows,
// which hides the latency of an iteration better than 4 waves of R rows:
// host-paced, every shape was faster at every scale of a 1920x1080 pyramid
// (e.g. (4,4) at 480x270: 5.22 -> 4.87 us per iteration; (4,8) at 960x540:
// 9.29 -> 8.18 us).  OF_ITER_BOUNDS asks for 4 waves per SIMD (its second
// argument counts waves per SIMD, not workgroups per CU), 128 VGPRs, so that 2
// workgroups of 8 waves share a CU; all shapes but (8,8) fit without spills.
constexpr int kIterWaves = 8;
// The lockstep batch kernel keeps 4 waves of R rows: with 8 waves of R/2 the
// batch of 64 mixed-size pairs took 79.0 ms instead of 75.7 ms (same box).
constexpr int kLsWaves = 4;
// __launch_bounds__(threads, minimum waves per SIMD)
// Square tiles of 16 waves with 3 iterations: 8, i.e. two workgroups per CU.
#define OF_ITER_BOUNDS(NW, K) \
    __launch_bounds__(64 * (NW), (NW) == 4 ? kIterBlocksPerCU : (NW) == 16 && (K) == 3 ? 8 : (K) == 8 ? 2 : 4)

// ---------------------------------------------------------------------------
// launch-per-chunk driver
// ---------------------------------------------------------------------------

// Stopping rule, evaluated by the last workgroup to finish: when the first
// iteration that meets it falls inside the launch before its last
// iteration, the launch's output is discarded and the next launch re-runs
// exactly that many iterations from the same input buffer.
template <int K, int R, int NW = 4, int T = 0>
__global__ OF_ITER_BOUNDS(NW, K) void k_tvl1_iter(IterArgs a)
{
    __shared__ TileSharedN<NW> sh;
    __shared__ SqShared<T ? T : 1> sh_sq;
    __shared__ double sh_err[NW][K];
    __shared__ double sh_tot[K];
    __shared__ double sh4[K * NW];
    __shared__ int sh_last;

    TvCtl* ctl = a.ctl;
    if (ctl->stop) return;
    const int cur = uniform(ctl->cur[a.level]);
    const int redo = uniform(ctl->redo);
    const int n0 = uniform(ctl->n);
    int kk = redo ? redo : a.max_iter - n0;
    if (kk > K) kk = K;
    if (kk <= 0) return;

    NoSync no_sync;
    double acc[K];
#pragma unroll
    for (int t = 0; t < K; t++) acc[t] = 0.0;
    if constexpr (T != 0) tile_iterate_sq<T, K, false>(a, blockIdx.x, blockIdx.y, cur, kk, acc, sh_sq, no_sync);
    else tile_iterate<K, R, false, NW>(a, blockIdx.x, blockIdx.y, cur, kk, acc, sh, no_sync);

    const unsigned nblocks = gridDim.x * gridDim.y;
    const unsigned bid = blockIdx.y * gridDim.x + blockIdx.x;
    const double part = block_sum<K, NW>(acc, sh_err, threadIdx.x);
    // The partials are published with device-scope atomic stores, which are
    // written through to the point of coherence of all XCDs, and every wave
    // waits for their completion (s_waitcnt vmcnt(0)) before the counter
    // increment; the last workgroup reads them with device-scope atomic
    // loads.  A device-scope release fence would instead write back the
    // XCD's whole L2 at the end of every workgroup.
    if (threadIdx.x < (unsigned)kk)
        __hip_atomic_store(a.partials + (size_t)threadIdx.x * nblocks + bid, part, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (threadIdx.x == 0) sh_last = atomicAdd(&ctl->counter, 1u) == nblocks - 1;
    __syncthreads();
    if (!sh_last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    grid_sums<K, NW>(a.partials, nblocks, kk, sh4, sh_tot);
    if (a.err_log && threadIdx.x < (unsigned)kk) a.err_log[n0 + threadIdx.x] = sh_tot[threadIdx.x];
    if (threadIdx.x == 0) {
        int n = n0, stop = 0, nredo = 0, flip = 0;
        if (redo) {
            n = n0 + redo;
            stop = 1;
            flip = 1;
        } else {
            const int keep = stop_after(sh_tot, kk, n0, a);
            if (keep == kk || keep == 0) {
                n = n0 + kk;
                flip = 1;
                stop = keep != 0;
            } else {
                nredo = keep;
            }
        }
        ctl->n = n;
        ctl->redo = nredo;
        ctl->stop = stop;
        if (flip) ctl->cur[a.level] = cur ^ 1;
        if (stop) *a.iters_slot = n;
        ctl->counter = 0;
        ctl->launches = ctl->launches + 1;
        const unsigned wl = ctl->wlaunches + 1;
        ctl->wlaunches = wl;
        const unsigned long long word = ((unsigned long long)a.epoch << 32) |
                                        ((unsigned long long)stop << 31) |
                                        (unsigned long long)(wl & 0x7FFFFFFFu);
        // the host only reads this word itself: no ordering with other data
        if (a.host_status)
            __hip_atomic_store(a.host_status, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---------------------------------------------------------------------------
// persistent driver
// ---------------------------------------------------------------------------

// Residency bound of a first grid barrier: `ticks` > 0 is the wall-clock
// time (ticks of the device's constant-rate clock) that a workgroup waits for the others
// before it reports kBarNotResident; `force` reports it at once (test hook).
struct FirstBound {
    unsigned long long ticks;
    int force;
};

__device__ __forceinline__ bool past_first_bound(const FirstBound& fb, unsigned long long t_end,
                                                 unsigned spins, TvCtl* ctl)
{
    if (!fb.ticks || (spins & 15u) != 0 || (unsigned long long)wall_clock64() < t_end) return false;
    __hip_atomic_store(&ctl->error, kBarNotResident, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// Grid barrier over `nb` co-resident workgroups.  Every wave first waits for
// its own memory operations to complete, so all state written by the
// workgroup (device-scope stores) is visible at the point of coherence before
// the arrival.  The wait is bounded: past ~1 s of polls it flags kBarTimeout
// and returns false, and the kernel ends; with a FirstBound it also ends
// after fb.ticks of wall-clock time with kBarNotResident.
__device__ __forceinline__ bool grid_barrier(TvCtl* ctl, unsigned nb, unsigned& gen, int* sh_ok,
                                             FirstBound fb = {0ull, 0})
{
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (threadIdx.x == 0) {
        int ok = 1;
        const unsigned g = gen;
        if (fb.force)
            __hip_atomic_store(&ctl->error, kBarNotResident, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long t_end = fb.ticks ? (unsigned long long)wall_clock64() + fb.ticks : 0ull;
        const unsigned old =
            __hip_atomic_fetch_add(&ctl->bar_count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (old == nb - 1) {
            __hip_atomic_store(&ctl->bar_count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_s_waitcnt(0);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __hip_atomic_store(&ctl->bar_gen, g + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            unsigned spins = 0;
            while (__hip_atomic_load(&ctl->bar_gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == g) {
                __builtin_amdgcn_s_sleep(2);
                if (++spins > (1u << 21)) {
                    __hip_atomic_store(&ctl->error, kBarTimeout, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
                    ok = 0;
                    break;
                }
                if (past_first_bound(fb, t_end, spins, ctl)) {
                    ok = 0;
                    break;
                }
                // another workgroup gave up: stop waiting too
                if ((spins & 1023u) == 0 &&
                    __hip_atomic_load(&ctl->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                    ok = 0;
                    break;
                }
            }
        }
        if (__hip_atomic_load(&ctl->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) ok = 0;
        gen = g + 1;
        *sh_ok = ok;
    }
    __syncthreads();
    return uniform(*sh_ok) != 0;
}

// Two-level grid barrier, for grids of many workgroups (the square-tile
// warping kernel: one workgroup per 8x8 centre).  Workgroup b arrives on the
// counter of group b % 8; the last arrival of a group arrives on the top
// counter; the last top arrival releases the group leaders, each leader its
// group.  With all workgroups arriving together a flat counter took ~10 us
// per barrier at 768 workgroups, the two levels ~3 us.  Each last arriver
// resets its counter and waits for the reset before it releases anyone; the
// release words only grow, and `ep` holds their values read at kernel start
// plus the barriers passed.  Bounded as grid_barrier.
struct BarEpoch {
    unsigned top, grp;
};

__device__ __forceinline__ bool bar_wait(const unsigned* w, unsigned target, TvCtl* ctl,
                                         const FirstBound& fb, unsigned long long t_end)
{
    unsigned spins = 0;
    while ((int)(__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - target) < 0) {
        __builtin_amdgcn_s_sleep(2);
        if (++spins > (1u << 21)) {
            __hip_atomic_store(&ctl->error, kBarTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        if (past_first_bound(fb, t_end, spins, ctl)) return false;
        if ((spins & 1023u) == 0 &&
            __hip_atomic_load(&ctl->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return false;
    }
    return true;
}

__device__ __forceinline__ bool grid_barrier2(TvCtl* ctl, unsigned nb, BarEpoch& ep, int* sh_ok,
                                              FirstBound fb = {0ull, 0})
{
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __syncthreads();
    if (threadIdx.x == 0) {
        if (fb.force)
            __hip_atomic_store(&ctl->error, kBarNotResident, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long t_end = fb.ticks ? (unsigned long long)wall_clock64() + fb.ticks : 0ull;
        const unsigned g = blockIdx.x % kBarGroups;
        const unsigned members = nb / kBarGroups + (g < nb % kBarGroups ? 1u : 0u);
        const unsigned groups = nb < (unsigned)kBarGroups ? nb : (unsigned)kBarGroups;
        unsigned* gc = &ctl->grp_count[g].v;
        unsigned* gg = &ctl->grp_gen[g].v;
        int ok = 1;
        const unsigned old = __hip_atomic_fetch_add(gc, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (old == members - 1) {
            __hip_atomic_store(gc, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned t =
                __hip_atomic_fetch_add(&ctl->bar_count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (t == groups - 1) {
                __hip_atomic_store(&ctl->bar_count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __builtin_amdgcn_s_waitcnt(0);
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                __hip_atomic_store(&ctl->bar_gen, ep.top + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else {
                ok = bar_wait(&ctl->bar_gen, ep.top + 1, ctl, fb, t_end);
            }
            if (ok) {
                __builtin_amdgcn_s_waitcnt(0);
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                __hip_atomic_store(gg, ep.grp + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else {
            ok = bar_wait(gg, ep.grp + 1, ctl, fb, t_end);
        }
        ep.top++;
        ep.grp++;
        if (fb.force) ok = 0;
        *sh_ok = ok;
    }
    __syncthreads();
    return uniform(*sh_ok) != 0;
}

// A whole warping: chunks of K iterations over all tiles (workgroup b takes
// tiles b, b+nb, ...), a grid barrier, then every workgroup sums the chunk's
// per-workgroup error partials in the same fixed order and takes the same
// stopping decision.  A stop inside a chunk re-runs exactly that many
// iterations from the chunk's input buffer.  The state is read and written
// with device-scope atomic accesses so that halos written by workgroups on
// other XCDs are seen without cache maintenance.  Partials are
// double-buffered by chunk parity.
template <int K, int R, int NW = 4, int T = 0>
__global__ OF_ITER_BOUNDS(NW, K) void k_tvl1_persist(IterArgs a, unsigned tiles_x, unsigned ntiles)
{
    __shared__ TileSharedN<NW> sh;
    __shared__ SqShared<T ? T : 1> sh_sq;
    __shared__ double sh_err[NW][K];
    __shared__ double sh_tot[K];
    __shared__ double sh4[K * NW];
    __shared__ int sh_ok;

    TvCtl* ctl = a.ctl;
    const unsigned nb = gridDim.x;
    unsigned gen = 0;
    BarEpoch ep{0u, 0u};
    if (threadIdx.x == 0) {
        gen = __hip_atomic_load(&ctl->bar_gen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ep.top = gen;
        ep.grp = __hip_atomic_load(&ctl->grp_gen[blockIdx.x % kBarGroups].v, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    }
    int cur = uniform(ctl->cur[a.level]);
    int n = 0;
    int redo = 0;
    int parity = 0;
    // the first barrier of a plain launch also checks that the grid is resident
    FirstBound fb{a.resident_ticks, a.force_not_resident};
    NoSync no_sync;
    while (true) {
        int kk = redo ? redo : a.max_iter - n;
        if (kk > K) kk = K;
        if (kk <= 0) break;
        double acc[K];
#pragma unroll
        for (int t = 0; t < K; t++) acc[t] = 0.0;
        for (unsigned tile = blockIdx.x; tile < ntiles; tile += nb)
            if constexpr (T != 0)
                tile_iterate_sq<T, K, true>(a, (int)(tile % tiles_x), (int)(tile / tiles_x), cur, kk, acc, sh_sq, no_sync);
            else
                tile_iterate<K, R, true, NW>(a, (int)(tile % tiles_x), (int)(tile / tiles_x), cur, kk, acc, sh, no_sync);
        if (redo) {   // the re-run chunk is final: no decision needed
            n += redo;
            cur ^= 1;
            break;
        }
        const double part = block_sum<K, NW>(acc, sh_err, threadIdx.x);
        double* pp = a.partials + (size_t)parity * K * nb;
        if (threadIdx.x < (unsigned)kk)
            __hip_atomic_store(pp + (size_t)threadIdx.x * nb + blockIdx.x, part, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        // square tiles run one workgroup per small tile: many workgroups
        if (!(T != 0 ? grid_barrier2(ctl, nb, ep, &sh_ok, fb) : grid_barrier(ctl, nb, gen, &sh_ok, fb)))
            return;
        fb = FirstBound{0ull, 0};
        grid_sums<K, NW>(pp, nb, kk, sh4, sh_tot);
        const int keep = uniform(stop_after(sh_tot, kk, n, a));
        if (a.err_log && blockIdx.x == 0 && threadIdx.x < (unsigned)kk)
            a.err_log[n + threadIdx.x] = sh_tot[threadIdx.x];
        parity ^= 1;
        if (keep == 0) {
            n += kk;
            cur ^= 1;
            continue;
        }
        if (keep == kk) {
            n += kk;
            cur ^= 1;
            break;
        }
        redo = keep;   // state of buffer `cur` is unchanged: re-run `keep` iterations
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctl->cur[a.level] = cur;
        ctl->n = n;
        ctl->stop = 1;
        *a.iters_slot = n;
    }
}

// ---------------------------------------------------------------------------
// neighbour-synchronised persistent driver
// ---------------------------------------------------------------------------

// Bounded wait of one wave until every lane's 64-bit word at `w` (lanes with a
// null pointer have none) reaches `want`; the words only grow within a
// warping.  Returns 1 then, 2 once the referee has published that the
// warping stops, 0 after flagging kBarTimeout past ~1 s of polls, after the
// first bound (kBarNotResident), or once another workgroup has flagged an
// error.
__device__ __forceinline__ int wave_wait(const IterArgs& a, const unsigned long long* w,
                                         unsigned long long want, const FirstBound& fb)
{
    TvCtl* ctl = a.ctl;
    const unsigned long long t_end = fb.ticks ? (unsigned long long)wall_clock64() + fb.ticks : 0ull;
    if (fb.force) {
        __hip_atomic_store(&ctl->error, kBarNotResident, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return 0;
    }
    unsigned spins = 0;
    while (true) {
        const bool wait = w && __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < want;
        if (!__any(wait)) return 1;
        if ((spins & 3u) == 3u) {
            bool stopped = false;
            if ((threadIdx.x & 63) < 2) {
                const unsigned long long d = __hip_atomic_load(&ctl->decision[threadIdx.x & 1].v,
                                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                stopped = (d >> 24) == a.seq && (d & 0xFull) != 0;
            }
            if (__any(stopped)) return 2;
        }
        __builtin_amdgcn_s_sleep(1);
        if (++spins > (1u << 21)) {
            __hip_atomic_store(&ctl->error, kBarTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return 0;
        }
        if (past_first_bound(fb, t_end, spins, ctl)) return 0;
        if ((spins & 1023u) == 0 &&
            __hip_atomic_load(&ctl->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return 0;
    }
}

// Bound of the wait for decision q: the first one checks that the referee is
// resident.  It decides once the slowest workgroup has completed the chunk:
// another 2 ms per 2^24 pixels, which take a chunk 0.3 ms.
__device__ __forceinline__ FirstBound referee_bound(const IterArgs& a, int q)
{
    if (q != 0) return FirstBound{0ull, 0};
    return FirstBound{a.resident_ticks + (a.resident_ticks * (unsigned long long)a.plane >> 24), a.force_not_resident};
}

// Synchronisation of one workgroup of k_tvl1_persist_nbr with the others.
// `stop_chunk`/`stop_keep`: set once the warping is known to stop after
// stop_keep iterations of chunk stop_chunk.  Members are uniform.
struct NbrSync {
    const IterArgs& a;
    // a plain launch also checks that the grid is resident: the first wait for
    // the neighbours (fb), and the one for the referee's first decision
    FirstBound fb;
    int* sh;         // LDS word for results of wave 0
    unsigned tiles_x, tiles_y, tile;
    int c;           // chunk of the current tile
    int seen;        // decisions up to this chunk are known to continue
    int stop_chunk, stop_keep;
    bool failed;
    bool rerun;      // the last pass: no waits, every tile is stored

    // Result of wave 0's wait, in every thread.  The first barrier also
    // orders the waits of a workgroup's earlier LDS reads of the word.
    __device__ __forceinline__ int share(int r)
    {
        __syncthreads();
        if (threadIdx.x == 0) *sh = r;
        __syncthreads();
        return uniform(*sh);
    }

    __device__ __forceinline__ int wait(const unsigned long long* w, unsigned long long want)
    {
        const int r = share(threadIdx.x < 64 ? wave_wait(a, w, want, fb) : 0);
        fb = FirstBound{0ull, 0};
        return r;
    }

    // Decision of chunk q once published: keep, or -1 if the wait failed.
    __device__ __forceinline__ int decision(int q)
    {
        int r = -1;
        if (threadIdx.x < 64) {
            const unsigned long long* w = &a.ctl->decision[q & 1].v;
            const unsigned long long want = (a.seq << 24) | ((unsigned long long)(q + 1) << 4);
            if (wave_wait(a, threadIdx.x == 0 ? w : nullptr, want, referee_bound(a, q)))
                r = (int)(__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xFull);
        }
        return share(r);
    }

    // The published stop (chunk, keep), if any.
    __device__ __forceinline__ void read_stop()
    {
        for (int q = 0; q < 2; q++) {
            unsigned long long d = 0ull;
            if (threadIdx.x == 0)
                d = __hip_atomic_load(&a.ctl->decision[q].v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const int r = share((int)((d >> 24) == a.seq ? (unsigned)(d & 0xFFFFFFull) : 0u));
            if (r & 15) {
                stop_chunk = (r >> 4) - 1;
                stop_keep = r & 15;
            }
        }
    }

    // The tile may start chunk c once its (up to) 8 neighbours have completed
    // chunk c-1: its extended tile reads their centres, and its stores
    // overwrite values their chunk c-1 read.  Lanes 0..8 poll one tile each.
    __device__ __forceinline__ bool ready()
    {
        if (c == 0 || rerun) return true;
        const unsigned long long* w = nullptr;
        if (threadIdx.x < 9 && threadIdx.x != 4) {
            const int x = (int)(tile % tiles_x) + (int)(threadIdx.x % 3) - 1;
            const int y = (int)(tile / tiles_x) + (int)(threadIdx.x / 3) - 1;
            if (x >= 0 && y >= 0 && x < (int)tiles_x && y < (int)tiles_y)
                w = a.tile_flags + (size_t)y * tiles_x + x;
        }
        const int r = wait(w, (a.seq << 20) | (unsigned)c);
        if (r == 2) read_stop();
        failed |= r == 0;
        return r == 1;
    }

    // Decision c-1 before a store of chunk c: false discards the tile.
    __device__ __forceinline__ bool store()
    {
        if (c == 0 || seen >= c - 1 || rerun) return true;
        const int r = decision(c - 1);
        failed |= r < 0;
        if (r < 0) return false;
        if (r) {
            stop_chunk = c - 1;
            stop_keep = r;
            return false;
        }
        seen = c - 1;
        return true;
    }

    // Past the last chunk: its decision stops the warping.
    __device__ __forceinline__ void last(int nchunks)
    {
        const int r = decision(nchunks - 1);
        failed |= r < 0;
        stop_chunk = nchunks - 1;
        stop_keep = r;
    }
};

// A whole warping without grid barriers.  Workgroups 0..nbw-1 iterate tiles
// (workgroup b takes tiles b, b+nbw, ...); a tile starts chunk c as soon as
// its neighbours have completed chunk c-1 (per-tile flags), so no workgroup
// waits for the whole grid.  Workgroup nbw is the referee: once every
// workgroup has completed its last tile of chunk c it sums their error
// partials in the fixed order of the barrier kernel, applies the stopping
// rule and publishes the decision.  Tiles do not wait for it: they iterate
// chunk c+1 from chunk c's output and check decision c before their first
// store of chunk c+1.  "Continue": they store as usual.  "Stop after keep
// iterations": they discard chunk c+1, and if keep is short of chunk c's
// length they re-run keep iterations from chunk c's input, which no store of
// chunk c+1 has touched.  Same arithmetic, partial sums and decisions as
// k_tvl1_persist, so the same bits and iteration counts.
// What a chunk costs beyond its arithmetic is the round trip to the neighbours
// (stores, flag, flag read, loads) and the scalar work around it: one wave
// polls for the workgroup, the warping's constants are loaded before the wait,
// everything uniform stays in scalar registers.  With the shorter dual update,
// 1920x1080 per scale (ms per solve): 2.12 -> 2.03, 960x540 (4,8) 1.04 ->
// 0.96..0.99, 480x270 0.67 -> 0.63, 240x135 (4,4) 0.56 -> 0.54, 120x68 0.40
// -> 0.32.  Dealing tiles to workgroups in rotation, so that all get the same
// number, was 5% slower at 1920x1080: two workgroups with 2 and 3 tiles
// already share a CU evenly.
template <int K, int R, int NW = 4, int T = 0>
__global__ OF_ITER_BOUNDS(NW, K) void k_tvl1_persist_nbr(IterArgs a, unsigned tiles_x, unsigned ntiles)
{
    static_assert(T ? (T - 2 * K >= K) : (NW * R - 2 * K >= K && 64 - 2 * K >= K),
                  "the halo of a tile must lie within its neighbours");
    __shared__ TileSharedN<NW> sh;
    __shared__ SqShared<T ? T : 1> sh_sq;
    __shared__ double sh_err[NW][K];
    __shared__ double sh_tot[K];
    __shared__ int sh_word;

    TvCtl* ctl = a.ctl;
    const unsigned nbw = gridDim.x - 1;   // tile workgroups; the last one is the referee
    const int cur0 = uniform(ctl->cur[a.level]);
    const int nchunks = (a.max_iter + K - 1) / K;

    if (blockIdx.x == nbw) {   // referee
        if (a.referee_absent) return;
        int n = 0, c = 0;
        while (c < nchunks) {
            const int kk = min(K, a.max_iter - n);
            const double* pp = a.partials + (size_t)(c & 1) * K * nbw;
            const unsigned long long want = (a.seq << 20) | (unsigned)(c + 1);
            double s[K];
#pragma unroll
            for (int t = 0; t < K; t++) s[t] = 0.0;
            bool ok = true;
            for (unsigned j0 = threadIdx.x & ~63u; j0 < nbw && ok; j0 += 64 * NW) {
                const unsigned j = j0 + (threadIdx.x & 63);   // workgroup
                const bool mine = j < nbw;
                const unsigned last = mine ? j + (ntiles - 1 - j) / nbw * nbw : 0u;
                ok = wave_wait(a, mine ? a.tile_flags + last : nullptr, want, FirstBound{0ull, 0}) == 1;
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
                if (ok && mine) {
#pragma unroll
                    for (int t = 0; t < K; t++)
                        if (t < kk)
                            s[t] += __hip_atomic_load(pp + (size_t)t * nbw + j, __ATOMIC_RELAXED,
                                                      __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            if (!uniform(__syncthreads_and(ok))) return;
            const double v = block_sum<K, NW>(s, sh_err, threadIdx.x);
            if (threadIdx.x < (unsigned)K) sh_tot[threadIdx.x] = v;
            __syncthreads();
            const int keep = uniform(stop_after(sh_tot, kk, n, a));
            if (a.err_log && threadIdx.x < (unsigned)kk) a.err_log[n + threadIdx.x] = sh_tot[threadIdx.x];
            if (threadIdx.x == 0)
                __hip_atomic_store(&ctl->decision[c & 1].v,
                                   (a.seq << 24) | ((unsigned long long)(c + 1) << 4) |
                                       (unsigned long long)keep,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            n += keep ? keep : kk;
            c++;
            if (keep) break;
            __syncthreads();   // sh_tot is rewritten next chunk
        }
        if (threadIdx.x == 0) {
            ctl->cur[a.level] = cur0 ^ (c & 1);
            ctl->n = n;
            ctl->stop = 1;
            *a.iters_slot = n;
        }
        return;
    }

    NbrSync sync{a, FirstBound{a.resident_ticks, a.force_not_resident}, &sh_word, tiles_x, ntiles / tiles_x,
                 0, 0, -1, 0, 0, false, false};
    double acc[K];
    // chunk after chunk; the last pass re-runs part of the chunk that stopped
    while (true) {
        if (!sync.stop_keep && sync.c >= nchunks) {
            if (nchunks == 0) return;
            sync.last(nchunks);
        }
        if (sync.failed) return;
        if (sync.stop_keep) {
            // the warping stopped after stop_keep iterations of chunk
            // stop_chunk: if that is short of the chunk, re-run them from its
            // input into its output
            if (sync.rerun || sync.stop_keep >= min(K, a.max_iter - sync.stop_chunk * K)) return;
            sync.rerun = true;
            sync.c = sync.stop_chunk;
        }
        const int c = sync.c, cur = cur0 ^ (c & 1);
        const int kk = sync.rerun ? sync.stop_keep : min(K, a.max_iter - c * K);
#pragma unroll
        for (int t = 0; t < K; t++) acc[t] = 0.0;
        for (unsigned tile = blockIdx.x; tile < ntiles; tile += nbw) {
            sync.tile = tile;
            const int bx = (int)(tile % tiles_x), by = (int)(tile / tiles_x);
            if constexpr (T != 0) tile_iterate_sq<T, K, true>(a, bx, by, cur, kk, acc, sh_sq, sync);
            else tile_iterate<K, R, true, NW>(a, bx, by, cur, kk, acc, sh, sync);
            if (sync.rerun) continue;
            if (sync.failed || sync.stop_keep) break;
            // after the workgroup's last tile of the chunk, its error partials
            // go out with the tile's stores; the flag once both have completed
            if (tile + nbw >= ntiles) {
                const double part = block_sum<K, NW>(acc, sh_err, threadIdx.x);
                if (threadIdx.x < (unsigned)kk)
                    __hip_atomic_store(a.partials + ((size_t)(c & 1) * K + threadIdx.x) * nbw + blockIdx.x, part,
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __builtin_amdgcn_s_waitcnt(0);
            __atomic_signal_fence(__ATOMIC_SEQ_CST);
            __syncthreads();
            if (threadIdx.x == 0)
                __hip_atomic_store(a.tile_flags + tile, (a.seq << 20) | (unsigned)(c + 1), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        sync.c++;
    }
}

// ---------------------------------------------------------------------------
// neighbour-synchronised driver with tagged values
// ---------------------------------------------------------------------------

// The state of one pixel.
struct SqState {
    float u1, u2, p11, p12, p21, p22;
    __device__ __forceinline__ void get(const SqPixel& q)
    {
        u1 = q.u1, u2 = q.u2, p11 = q.p11, p12 = q.p12, p21 = q.p21, p22 = q.p22;
    }
    __device__ __forceinline__ void put(SqPixel& q) const
    {
        q.u1 = u1, q.u2 = u2, q.p11 = p11, q.p12 = p12, q.p21 = p21, q.p22 = p22;
    }
};

// A 32-bit value and its tag in one word: whoever reads the tag has the value.
__device__ __forceinline__ void st_tagged(unsigned long long* w, unsigned tag, unsigned v)
{
    __hip_atomic_store(w, ((unsigned long long)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Bounded wait of one wave until the N words at w, w + stride, .. of every lane
// with `need` carry `tag`; v receives their values.  The bounds are wave_wait's;
// false after flagging an error or once another workgroup has flagged one.
template <int N>
__device__ __forceinline__ bool wait_tagged(const IterArgs& a, const unsigned long long* w, size_t stride, int n,
                                            bool need, unsigned tag, unsigned (&v)[N], const FirstBound& fb)
{
    TvCtl* ctl = a.ctl;
    if (fb.force) {
        __hip_atomic_store(&ctl->error, kBarNotResident, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return false;
    }
    const unsigned long long t_end = fb.ticks ? (unsigned long long)wall_clock64() + fb.ticks : 0ull;
    unsigned spins = 0;
    while (true) {
        bool there = true;
        if (need) {
            unsigned long long x[N];
#pragma unroll
            for (int i = 0; i < N; i++)
                if (i < n) x[i] = __hip_atomic_load(w + i * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int i = 0; i < N; i++)
                if (i < n) {
                    there &= (unsigned)(x[i] >> 32) == tag;
                    v[i] = (unsigned)x[i];
                }
        }
        if (__all(there)) return true;
        __builtin_amdgcn_s_sleep(1);
        if (++spins > (1u << 21)) {
            __hip_atomic_store(&ctl->error, kBarTimeout, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        if (past_first_bound(fb, t_end, spins, ctl)) return false;
        if ((spins & 1023u) == 0 &&
            __hip_atomic_load(&ctl->error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            return false;
    }
}

// A whole warping on square tiles that all have a workgroup of their own
// (blockIdx = tile, the last block is the referee).  The protocol and the
// decisions are k_tvl1_persist_nbr's, the synchronisation is in the data: a
// tile keeps its pixels in registers and stores only the ring that its
// neighbours read, each value in one word with the tag tag0 + chunk + 1; they
// wait for the words themselves.  No store is waited for and no flag follows
// it.  Error partials go to the referee the same way.
// Both parities of a word are safe to reuse: a tile stores chunk c after it has
// read its neighbours' chunk c-1, which they stored after reading its chunk
// c-2; partials and decisions likewise, since a tile sees decision c-2 before
// it iterates chunk c.  By then it has chunk c-1's output in registers, and
// keeps the inputs of chunks c-1 and c-2: "continue" goes on, "stop after keep
// iterations of chunk c-2" takes chunk c-1's input or re-runs keep iterations
// from chunk c-2's.  A tile never waits on work that waits on it, so no order of
// the workgroups deadlocks, and the waits are bounded all the same.
// Bound by the chain of an iteration and the exchange, about 3 us per chunk
// where stores, flag and loads one after the other took 4.5.  Whole scales, ms:
// 480x270 0.515 -> 0.464, 240x135 0.386 -> 0.349, 120x68 0.292 -> 0.257, 40x30 0.360
// -> 0.307.  Four iterations per chunk instead of five, and polling without
// sleeps, change no scale by more than 3%.
template <int T, int K>
__global__ OF_ITER_BOUNDS(T * T / 64, K) void k_tvl1_persist_tag(IterArgs a, unsigned tiles_x, unsigned ntiles)
{
    constexpr int NW = T * T / 64, C = T - 2 * K;
    static_assert(C >= K, "the halo of a tile must lie within its neighbours");
    static_assert(T * T > kSqOnePerCu && K <= kSqMaxIters, "the referee has a lane per tile");
    __shared__ SqShared<T> sh;
    __shared__ double sh_err[NW][K];
    __shared__ double sh_tot[K];
    __shared__ int sh_keep[2], sh_fail[2];

    TvCtl* ctl = a.ctl;
    const size_t plane = (size_t)a.plane;
    unsigned long long* const parts = a.halo + 12 * plane;   // [parity][iteration][half][tile]
    const int cur0 = uniform(ctl->cur[a.level]);
    const int nchunks = (a.max_iter + K - 1) / K;

    if (blockIdx.x == ntiles) {   // referee
        if (a.referee_absent) return;
        int n = 0, c = 0;
        while (c < nchunks) {
            const int kk = min(K, a.max_iter - n);
            const bool mine = threadIdx.x < ntiles;
            unsigned v[2 * K] = {};
            const bool ok = wait_tagged<2 * K>(a, parts + (size_t)(c & 1) * 2 * K * ntiles + threadIdx.x, ntiles,
                                               2 * kk, mine, a.tag0 + (unsigned)c + 1u, v, FirstBound{0ull, 0});
            if (!uniform(__syncthreads_and(ok))) return;
            double s[K];
#pragma unroll
            for (int t = 0; t < K; t++)
                s[t] = mine && t < kk ? __hiloint2double((int)v[2 * t + 1], (int)v[2 * t]) : 0.0;
            const double tot = block_sum<K, NW>(s, sh_err, threadIdx.x);
            if (threadIdx.x < (unsigned)K) sh_tot[threadIdx.x] = tot;
            __syncthreads();
            const int keep = uniform(stop_after(sh_tot, kk, n, a));
            if (a.err_log && threadIdx.x < (unsigned)kk) a.err_log[n + threadIdx.x] = sh_tot[threadIdx.x];
            if (threadIdx.x == 0)
                __hip_atomic_store(&ctl->decision[c & 1].v,
                                   (a.seq << 24) | ((unsigned long long)(c + 1) << 4) |
                                       (unsigned long long)keep,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            n += keep ? keep : kk;
            c++;
            if (keep) break;
            __syncthreads();   // sh_tot is rewritten next chunk
        }
        if (threadIdx.x == 0) {
            ctl->cur[a.level] = cur0 ^ 1;
            ctl->n = n;
            ctl->stop = 1;
            *a.iters_slot = n;
        }
        return;
    }

    const int bx = (int)(blockIdx.x % tiles_x), by = (int)(blockIdx.x / tiles_x);
    const int lx = threadIdx.x % T, ly = threadIdx.x / T;
    const int x = bx * C - K + lx, y = by * C - K + ly;
    const bool in = x >= 0 && x < a.nx && y >= 0 && y < a.ny;
    const bool centre = lx >= K && lx < K + C && ly >= K && ly < K + C;
    // neighbours read the K outermost pixels of the centre
    const bool ring = in && centre && (lx < 2 * K || lx >= C || ly < 2 * K || ly >= C);
    const size_t idx = (size_t)y * a.nx + x;
    SqPixel q;
    q.fc = x == 0;
    q.lc = x == a.nx - 1;
    q.fr = y == 0;
    q.lr = y == a.ny - 1;
    q.mine = in && centre;
    if (threadIdx.x < 2) sh_fail[threadIdx.x] = 0;
    sq_load_constants(a, q, in, idx);
    sq_load_state<false>(a, q, in, idx, cur0);
    __syncthreads();

    // decision of chunk d, in wave 0: keep, or -1 if the wait failed.  The
    // first wait for the neighbours (fb) and the one for the first decision
    // check that the grid is resident
    FirstBound fb{a.resident_ticks, a.force_not_resident};
    auto decision = [&](int d) -> int {
        const unsigned long long* w = &ctl->decision[d & 1].v;
        const unsigned long long want = (a.seq << 24) | ((unsigned long long)(d + 1) << 4);
        if (!wave_wait(a, threadIdx.x == 0 ? w : nullptr, want, referee_bound(a, d))) return -1;
        return uniform((int)(__hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xFull));
    };
    SqState in0{}, in1{};   // inputs of the chunks before the last and last iterated
    double acc[K];
    int c = 0, keep = 0, full = 0;   // the warping stops after `keep` of the `full` iterations of a chunk
    while (true) {
        if (c > 0) {
            bool ok = true;
            if (c < nchunks) {
                const size_t par = (size_t)((c - 1) & 1) * 6 * plane;
                unsigned v[6] = {};
                const bool need = in && !centre;
                ok = wait_tagged<6>(a, a.halo + par + (need ? idx : 0), plane, 6, need, a.tag0 + (unsigned)c, v, fb);
                if (need) {
                    q.u1 = __uint_as_float(v[0]);
                    q.u2 = __uint_as_float(v[1]);
                    q.p11 = __uint_as_float(v[2]);
                    q.p12 = __uint_as_float(v[3]);
                    q.p21 = __uint_as_float(v[4]);
                    q.p22 = __uint_as_float(v[5]);
                }
            }
            if (threadIdx.x < 64) {
                int r = 0;
                if (ok && c > 1) r = decision(c - 2);
                if (threadIdx.x == 0) sh_keep[c & 1] = r;
                ok &= r >= 0;
            }
            if (!ok) sh_fail[c & 1] = 1;
            fb = FirstBound{0ull, 0};   // the first wait was it
            __syncthreads();
            if (uniform(sh_fail[c & 1])) return;
            keep = uniform(sh_keep[c & 1]);
            if (keep) {   // chunk c-2: in0 is its input, in1 its output
                full = min(K, a.max_iter - (c - 2) * K);
                break;
            }
            if (c == nchunks) break;
        }
        in0 = in1;
        in1.get(q);
        const int kk = min(K, a.max_iter - c * K);
#pragma unroll
        for (int t = 0; t < K; t++) acc[t] = 0.0;
        sq_iterations<T, K>(a, q, kk, T, acc, sh);
        const unsigned tag = a.tag0 + (unsigned)c + 1u;
        if (ring && c + 1 < nchunks) {
            unsigned long long* w = a.halo + (size_t)(c & 1) * 6 * plane + idx;
            st_tagged(w, tag, __float_as_uint(q.u1));
            st_tagged(w + plane, tag, __float_as_uint(q.u2));
            st_tagged(w + 2 * plane, tag, __float_as_uint(q.p11));
            st_tagged(w + 3 * plane, tag, __float_as_uint(q.p12));
            st_tagged(w + 4 * plane, tag, __float_as_uint(q.p21));
            st_tagged(w + 5 * plane, tag, __float_as_uint(q.p22));
        }
        const double part = block_sum<K, NW>(acc, sh_err, threadIdx.x);
        if (threadIdx.x < (unsigned)kk) {
            unsigned long long* w = parts + ((size_t)(c & 1) * 2 * K + 2 * threadIdx.x) * ntiles + blockIdx.x;
            st_tagged(w, tag, (unsigned)__double2loint(part));
            st_tagged(w + ntiles, tag, (unsigned)__double2hiint(part));
        }
        c++;
    }
    if (!keep) {   // the last chunk's decision: in1 is its input, q holds its output
        if (threadIdx.x < 64) {
            const int r = decision(nchunks - 1);
            if (threadIdx.x == 0) sh_keep[(c + 1) & 1] = r;
        }
        __syncthreads();
        keep = uniform(sh_keep[(c + 1) & 1]);
        if (keep < 0) return;
        full = a.max_iter - (nchunks - 1) * K;
        in0 = in1;
        in1.get(q);
    }
    if (keep < full) {
        in0.put(q);
        sq_iterations<T, K>(a, q, keep, T, acc, sh);
    } else {
        in1.put(q);
    }
    if (q.mine) sq_store_state<false>(a, q, idx, cur0 ^ 1);
}

// ---------------------------------------------------------------------------
// one-workgroup driver
// ---------------------------------------------------------------------------

// A whole warping of a scale of at most 32 x 32 pixels in one workgroup of 32
// lanes per image row: the state stays in registers, no other workgroup takes
// part.  Chunks of K iterations; a stop inside a chunk re-runs that many from
// the state at its start.  Bound by the dependent chain of an iteration and its
// two exchanges (0.7 us at 15 rows); the neighbour kernel's chunks add their
// round trip through memory (20x15: 1.5 us per iteration).
constexpr int kSingleCols = 32;
template <int K>
__global__ __launch_bounds__(1024) void k_tvl1_single(IterArgs a)
{
    constexpr int T = kSingleCols;
    __shared__ SqShared<T> sh;
    __shared__ double sh_err[16][K];
    const int lx = threadIdx.x % T, ly = threadIdx.x / T;
    const int nx = a.nx, ny = a.ny;
    const int rows = blockDim.x / T, nw = blockDim.x / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool in = lx < nx && ly < ny;
    const size_t idx = (size_t)ly * nx + lx;
    const int cur = uniform(a.ctl->cur[a.level]);
    SqPixel q;
    q.fc = lx == 0;
    q.lc = lx == nx - 1;
    q.fr = ly == 0;
    q.lr = ly == ny - 1;
    q.mine = in;
    sq_load_constants(a, q, in, idx);
    sq_load_state<false>(a, q, in, idx, cur);
    int n = 0;
    while (n < a.max_iter) {
        const int kk = min(K, a.max_iter - n);
        const SqPixel start = q;
        double acc[K];
#pragma unroll
        for (int t = 0; t < K; t++) acc[t] = 0.0;
        sq_iterations<T, K>(a, q, kk, rows, acc, sh);
#pragma unroll
        for (int t = 0; t < K; t++) {
            const double v = wave_sum_f64(acc[t]);
            if (lane == 63) sh_err[wave][t] = v;
        }
        __syncthreads();
        double tot[K];
#pragma unroll
        for (int t = 0; t < K; t++) tot[t] = 0.0;
        for (int w = 0; w < nw; w++) {
#pragma unroll
            for (int t = 0; t < K; t++) tot[t] += sh_err[w][t];
        }
        if (a.err_log && threadIdx.x == 0) {
#pragma unroll
            for (int t = 0; t < K; t++)
                if (t < kk) a.err_log[n + t] = tot[t];
        }
        int keep = 0;
#pragma unroll
        for (int t = K - 1; t >= 0; t--)
            if (t < kk && !(tot[t] / (double)a.plane > a.eps2)) keep = t + 1;
        keep = uniform(keep);
        if (keep && keep < kk) {
            q = start;
            sq_iterations<T, K>(a, q, keep, rows, acc, sh);
        }
        n += keep ? keep : kk;
        if (keep) break;
        __syncthreads();   // sh_err is rewritten next chunk
    }
    if (n > 0 && in) sq_store_state<false>(a, q, idx, cur ^ 1);
    if (threadIdx.x == 0) {
        if (n > 0) a.ctl->cur[a.level] = cur ^ 1;
        a.ctl->n = n;
        a.ctl->stop = 1;
        *a.iters_slot = n;
    }
}

// ---------------------------------------------------------------------------
// lockstep driver: one scale of many pairs per launch
// ---------------------------------------------------------------------------

// Inclusive prefix sums of v[0..n), n <= kLsMaxPairs, by one workgroup of
// NT threads (Hillis-Steele over LDS).
template <int NT>
__device__ __forceinline__ void ls_block_scan(unsigned* v, int n)
{
    static_assert(kLsMaxPairs % NT == 0, "pairs per thread");
    constexpr int PER = kLsMaxPairs / NT;
    for (int off = 1; off < n; off <<= 1) {
        unsigned t[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int e = (int)threadIdx.x + NT * k;
            t[k] = (e < n && e >= off) ? v[e - off] : 0u;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int e = (int)threadIdx.x + NT * k;
            if (e < n) v[e] += t[k];
        }
        __syncthreads();
    }
}

// Iterations of one pair's tile `bid` (kk <= K of them) and, in the
// workgroup that finishes the pair's last tile of this launch, the pair's
// stopping decision: the same partial sums, order and rule as k_tvl1_iter.
template <int K, int R, int NW>
__device__ __forceinline__ void ls_tile(const LsPhase& ph, const LsPair* P, unsigned bid,
                                        TileSharedN<NW>& sh, double (*sh_err)[K], double* sh_tot,
                                        double* sh4, int* sh_last)
{
    // the table entry is read in place: a private copy would be indexed by
    // `cur` at run time and live in scratch memory
    const IterArgs& a = P->a;
    TvCtl* ctl = a.ctl;
    const int cur = uniform(ctl->cur[a.level]);
    const int redo = uniform(ctl->redo);
    const int n0 = uniform(ctl->n);
    int kk = redo ? redo : a.max_iter - n0;
    if (kk > K) kk = K;
    const unsigned nblocks = P->ntiles;
    NoSync no_sync;
    double acc[K];
#pragma unroll
    for (int t = 0; t < K; t++) acc[t] = 0.0;
    if (kk > 0) tile_iterate<K, R, false, NW>(a, (int)(bid % P->gx), (int)(bid / P->gx), cur, kk, acc, sh, no_sync);
    const double part = block_sum<K, NW>(acc, sh_err, threadIdx.x);
    if ((int)threadIdx.x < kk)
        __hip_atomic_store(a.partials + (size_t)threadIdx.x * nblocks + bid, part, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (threadIdx.x == 0) *sh_last = atomicAdd(&ctl->counter, 1u) == nblocks - 1;
    __syncthreads();
    if (*sh_last) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
        grid_sums<K, NW>(a.partials, nblocks, kk, sh4, sh_tot);
        if (threadIdx.x == 0) {
            int n = n0, stop = 0, nredo = 0, flip = 0;
            if (kk <= 0) {   // nothing left to do: only reached if the list was stale
                stop = 1;
            } else if (redo) {
                n = n0 + redo;
                stop = 1;
                flip = 1;
            } else {
                const int keep = stop_after(sh_tot, kk, n0, a);
                if (keep == kk || keep == 0) {
                    n = n0 + kk;
                    flip = 1;
                    stop = keep != 0;
                } else {
                    nredo = keep;
                }
            }
            ctl->n = n;
            ctl->redo = nredo;
            if (flip) ctl->cur[a.level] = cur ^ 1;
            if (stop)
                ph.iters[((size_t)P->pair_id * kMaxScales + a.level) * ph.warps + ph.warp] = n;
            ctl->counter = 0;
            ctl->launches = ctl->launches + 1;
            // read in this launch by the workgroup that rebuilds the work list
            __hip_atomic_store(&ctl->stop, stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    __syncthreads();
}

template <int K, int R, int NW>
__global__ OF_ITER_BOUNDS(NW, K) void k_ls_iter(LsPhase ph, const LsPair* __restrict__ pairs,
                                             LsCtl* mc, unsigned long long* host_status,
                                             unsigned epoch)
{
    // `pairs` is ph.pairs as a restrict kernel argument: the compiler may
    // then read the (wave-uniform) table entries with scalar loads
    constexpr int NT = 64 * NW;
    __shared__ TileSharedN<NW> sh;
    __shared__ double sh_err[NW][K];
    __shared__ double sh_tot[K];
    __shared__ double sh4[K * NW];
    __shared__ int sh_last;
    __shared__ unsigned s_pair[kLsMaxPairs], s_base[kLsMaxPairs];

    const unsigned nlist = mc->nlist;
    const unsigned ntot = mc->ntiles;
    for (unsigned k = threadIdx.x; k < nlist; k += NT) {
        s_pair[k] = mc->list_pair[k];
        s_base[k] = mc->list_base[k];
    }
    __syncthreads();
    for (unsigned t = blockIdx.x; t < ntot; t += gridDim.x) {
        int lo = 0, hi = (int)nlist - 1;   // last listed pair whose first entry is <= t
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (s_base[mid] <= t) lo = mid;
            else hi = mid - 1;
        }
        // the owner is the same in every lane: keep it (and the table entry's
        // fields) in scalar registers
        const unsigned pk = __builtin_amdgcn_readfirstlane(s_pair[lo]);
        const unsigned bid = __builtin_amdgcn_readfirstlane(t - s_base[lo]);
        ls_tile<K, R, NW>(ph, pairs + pk, bid, sh, sh_err, sh_tot, sh4, &sh_last);
    }

    // launch completion: the last workgroup rebuilds the work list
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (threadIdx.x == 0) sh_last = atomicAdd(&mc->counter, 1u) == gridDim.x - 1;
    __syncthreads();
    if (!sh_last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    const int np = ph.npairs;
    for (int k = threadIdx.x; k < np; k += NT) {
        const int stop =
            __hip_atomic_load(&ph.pairs[k].a.ctl->stop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_pair[k] = stop ? 0u : 1u;
        s_base[k] = stop ? 0u : ph.pairs[k].ntiles;
    }
    __syncthreads();
    ls_block_scan<NT>(s_pair, np);
    ls_block_scan<NT>(s_base, np);
    for (int k = threadIdx.x; k < np; k += NT) {
        const unsigned before = k ? s_pair[k - 1] : 0u;
        if (s_pair[k] != before) {   // pair k still iterates
            mc->list_pair[before] = (unsigned)k;
            mc->list_base[before] = k ? s_base[k - 1] : 0u;
        }
    }
    if (threadIdx.x == 0) {
        const unsigned left = np ? s_pair[np - 1] : 0u;
        mc->nlist = left;
        mc->ntiles = np ? s_base[np - 1] : 0u;
        mc->counter = 0;
        const unsigned done = mc->launches + 1;
        mc->launches = done;
        const unsigned long long word = ((unsigned long long)epoch << 32) |
                                        ((unsigned long long)(left == 0) << 31) |
                                        (unsigned long long)(done & 0x7FFFFFFFu);
        if (host_status)
            __hip_atomic_store(host_status, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------

bool iter_config_ok(int K, int R)
{
    if (R == 0) return K == 1 || K == 2 || K == 4;   // square tiles
    if (!(K == 1 || K == 2 || K == 4 || K == 8)) return false;
    if (!(R == 2 || R == 4 || R == 8)) return false;
    return 4 * R - 2 * K >= 4;
}

void iter_grid(int K, int R, int nx, int ny, unsigned* gx, unsigned* gy)
{
    if (R == 0) {   // square tiles
        *gx = cdiv((size_t)nx, (size_t)(kSqTile - 2 * K));
        *gy = cdiv((size_t)ny, (size_t)(kSqTile - 2 * K));
        return;
    }
    *gx = cdiv((size_t)nx, (size_t)(64 - 2 * K));
    *gy = cdiv((size_t)ny, (size_t)(4 * R - 2 * K));
}

template <int K, int R>
static hipError_t launch_kr(const IterArgs& a, hipStream_t s)
{
    unsigned gx, gy;
    iter_grid(K, R, a.nx, a.ny, &gx, &gy);
    if constexpr (R == 0)
        hipLaunchKernelGGL((k_tvl1_iter<K, 0, 4, kSqTile>), dim3(gx, gy), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((k_tvl1_iter<K, R * 4 / kIterWaves, kIterWaves>), dim3(gx, gy),
                           dim3(64 * kIterWaves), 0, s, a);
    return hipGetLastError();
}

int launch_iter(int K, int R, const IterArgs& a, hipStream_t s)
{
    hipError_t e = hipErrorInvalidValue;
#define OF_CASE(k, r) \
    if (K == k && R == r) e = launch_kr<k, r>(a, s);
    OF_CASE(1, 0) OF_CASE(2, 0) OF_CASE(4, 0)
    OF_CASE(1, 2) OF_CASE(2, 2)
    OF_CASE(1, 4) OF_CASE(2, 4) OF_CASE(4, 4)
    OF_CASE(1, 8) OF_CASE(2, 8) OF_CASE(4, 8) OF_CASE(8, 8)
#undef OF_CASE
    if (e != hipSuccess) {
        record_hip_error(e, "k_tvl1_iter launch", __FILE__, __LINE__);
        return OF_ERR_HIP;
    }
    return OF_OK;
}

// The persistent warping kernel of launch shape (K, R): 64 x 4R tiles as
// kIterWaves waves, or (R = 0) square tiles as 4 waves.
template <int K, int R, bool NBR>
static const void* persist_kernel()
{
    if constexpr (NBR) {
        if constexpr (R == 0) return (const void*)k_tvl1_persist_nbr<K, 0, 4, kSqTile>;
        else return (const void*)k_tvl1_persist_nbr<K, R * 4 / kIterWaves, kIterWaves>;
    } else {
        if constexpr (R == 0) return (const void*)k_tvl1_persist<K, 0, 4, kSqTile>;
        else return (const void*)k_tvl1_persist<K, R * 4 / kIterWaves, kIterWaves>;
    }
}

unsigned iter_tiles(int K, int R, int nx, int ny)
{
    unsigned gx, gy;
    iter_grid(K, R, nx, ny, &gx, &gy);
    return gx * gy;
}

template <int R>
static constexpr int persist_threads()
{
    return R == 0 ? 256 : 64 * kIterWaves;
}

// Launch mode of the persistent kernel.  It is launched as a plain kernel of
// a grid that fits the device at once (occupancy x CUs), which starts every
// workgroup when nothing else holds the CUs.  A cooperative launch would
// guarantee co-residency, but the runtime brackets it with about 11 us of
// idle device time on each side (kernel trace of the 1920x1080 solve, 20
// such launches per solve: 6.07 vs 5.67 ms per solve).  Instead the first
// grid barrier of each launch (with neighbour flags: each workgroup's first
// wait for its neighbours and its first for the referee, the last workgroup of
// the grid) checks residency with a wall-clock bound: if the grid did not
// fully start (another persistent kernel on another stream or process holding
// CUs, a CU-masked stream), the kernel ends with kBarNotResident, the host
// switches the process to host-paced launches for the warpings that would be
// persistent, and repeats the solve.  Host-paced launches need no
// co-residency and give the same bits.
static std::atomic<int> g_host_paced{-1};   // -1: not read from the environment yet
static std::atomic<int> g_force_not_resident{0}, g_referee_absent{0};
constexpr double kResidentBoundUs = 2000.0;   // first-barrier wait of a launch

bool persist_host_paced()
{
    int m = g_host_paced.load(std::memory_order_relaxed);
    if (m < 0) {
        const char* e = std::getenv("AMDFLOW_HOST_PACED");
        const int want = (e && e[0] == '1') ? 1 : 0;
        g_host_paced.compare_exchange_strong(m, want);
        m = g_host_paced.load(std::memory_order_relaxed);
    }
    return m == 1;
}

void set_persist_host_paced(bool on) { g_host_paced.store(on ? 1 : 0); }

void set_persist_force_not_resident(bool on) { g_force_not_resident.store(on ? 1 : 0); }

void set_persist_referee_absent(bool on) { g_referee_absent.store(on ? 1 : 0); }

static std::atomic<unsigned long long> g_warp_seq{0};

unsigned long long next_warp_seq() { return g_warp_seq.fetch_add(1) + 1; }

// Launches the persistent kernel `fn` of `threads` threads over gx x gy tiles.
// nbr: the neighbour-synchronised kernel with K iterations per chunk, whose
// grid is the tile workgroups plus one referee workgroup.  `cache` holds the
// kernel's co-resident workgroups on the device (-1: not known yet); solves of
// several threads may find it so at once, and then each asks.
// tile_each: every tile needs a workgroup of its own.
static int launch_persist_grid(const void* fn, int threads, int K, bool nbr, unsigned gx, unsigned gy,
                               const IterArgs& a, int nblocks, std::atomic<int>& cache, hipStream_t s,
                               bool tile_each = false)
{
    static std::atomic<unsigned long long> bound{0};   // written before any cache
    int resident = cache.load(std::memory_order_acquire);
    if (resident < 0) {
        int dev = 0, per_cu = 0, cus = 0, clock_khz = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            hipDeviceGetAttribute(&clock_khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess ||
            hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, 0) != hipSuccess) {
            (void)hipGetLastError();
            return OF_ERR_HIP;
        }
        // the residency bound in wall-clock ticks (at least 1 ms at any rate)
        bound.store((unsigned long long)(kResidentBoundUs * 1e-3 * std::max(clock_khz, 1000)),
                    std::memory_order_relaxed);
        // at most 4 workgroups per CU: 1024 arrivals on one counter and
        // pollers of one word per barrier are already plenty (the compiled
        // bound allows 2 of 8 waves)
        // a workgroup's waves are dealt to the 4 SIMDs from the first on: one of
        // 9 waves puts 3 on one SIMD, which the occupancy query does not see
        const int waves = threads / 64, per_simd = (waves + 3) / 4;
        per_cu = std::min(per_cu, per_cu * waves / 4 / per_simd);
        resident = std::min(per_cu, 4) * cus;
        cache.store(resident, std::memory_order_release);
    }
    if (resident <= (nbr ? 1 : 0)) return OF_ERR_UNSUPPORTED;
    const unsigned ntiles = gx * gy;
    unsigned nb = nblocks > 0 ? (unsigned)nblocks : ntiles;
    if (nb > ntiles) nb = ntiles;
    if (nb > (unsigned)resident - (nbr ? 1u : 0u)) nb = (unsigned)resident - (nbr ? 1u : 0u);
    if (tile_each && nb < ntiles) return OF_ERR_UNSUPPORTED;
    if (nbr) {
        if (!a.tile_flags || a.seq == 0 || a.seq >= kNbrMaxSeq) return OF_ERR_ARG;
        if ((long long)a.max_iter / K + 1 >= kNbrMaxChunks) return OF_ERR_UNSUPPORTED;
        nb += 1;   // the referee
    }
    IterArgs args = a;
    args.resident_ticks = bound.load(std::memory_order_relaxed);
    args.force_not_resident = g_force_not_resident.load(std::memory_order_relaxed);
    args.referee_absent = g_referee_absent.load(std::memory_order_relaxed);
    unsigned tx = gx, nt = ntiles;
    void* kargs[] = {(void*)&args, (void*)&tx, (void*)&nt};
    const hipError_t e = hipLaunchKernel(fn, dim3(nb), dim3(threads), kargs, 0, s);
    if (e != hipSuccess) {
        record_hip_error(e, "k_tvl1_persist launch", __FILE__, __LINE__);
        return OF_ERR_HIP;
    }
    return OF_OK;
}

template <int K, int R, bool NBR>
static int launch_persist_kr(const IterArgs& a, int nblocks, hipStream_t s)
{
    static std::atomic<int> resident{-1};
    unsigned gx, gy;
    iter_grid(K, R, a.nx, a.ny, &gx, &gy);
    return launch_persist_grid(persist_kernel<K, R, NBR>(), persist_threads<R>(), K, NBR, gx, gy, a, nblocks,
                               resident, s);
}

// Square tiles of T x T pixels with K iterations per chunk.
template <int T, int K>
static int launch_persist_sq(const IterArgs& a, int nblocks, hipStream_t s)
{
    static std::atomic<int> resident{-1};
    static_assert(T * T % 64 == 0 && T * T <= 1024, "whole waves");
    static_assert(K <= kSqMaxIters, "room for the partials");
    const unsigned gx = cdiv((size_t)a.nx, (size_t)(T - 2 * K)), gy = cdiv((size_t)a.ny, (size_t)(T - 2 * K));
    return launch_persist_grid((const void*)k_tvl1_persist_nbr<K, 0, T * T / 64, T>, T * T, K, true, gx, gy, a,
                               nblocks, resident, s);
}

// The same with tagged values; OF_ERR_UNSUPPORTED where the tiles do not all
// have a workgroup, or without the words for them.
template <int T, int K>
static int launch_persist_tagged(const IterArgs& a, int nblocks, hipStream_t s)
{
    static std::atomic<int> resident{-1};
    const unsigned gx = cdiv((size_t)a.nx, (size_t)(T - 2 * K)), gy = cdiv((size_t)a.ny, (size_t)(T - 2 * K));
    if (!a.halo || nblocks > 0) return OF_ERR_UNSUPPORTED;
    return launch_persist_grid((const void*)k_tvl1_persist_tag<T, K>, T * T, K, true, gx, gy, a, (int)(gx * gy),
                               resident, s, true);
}

// The shape (4, 0) with neighbour flags: square tiles of a size chosen by the
// scale's.  A chunk costs its iterations (one tile per CU: 0.5 us each at 16 x
// 16, 0.74 at 24 x 24, 0.9 at 32 x 32, the chain of an iteration and its two
// barriers) plus 4.5 us of exchange with the neighbours, so the line lies where
// the next smaller tile no longer has a CU of its own: within that, more
// iterations per chunk and smaller tiles win.  Whole scales, five warpings with
// their set-up, MI355X:
//    scale      16x16 K4   16x16 K5   24x24 K5   32x32 K5   32x32 K4   32x32 K3
//    80x60         0.31       0.29       0.33                             0.53   ms
//    120x68        0.31       0.30       0.37       0.47       0.47       0.55
//    161x120       0.36       0.41       0.33       0.40       0.41       0.46
//    240x135       0.44       0.57       0.37       0.44       0.47       0.55
//    321x240       0.53       0.58                  0.33       0.33       0.38
//    512x218       0.55       0.65                  0.32       0.35       0.38
//    480x270       0.78       1.03                  0.73       0.52       0.61
//    641x479       0.70       1.10                  0.60       0.58       0.44
//    1024x436      0.90       1.40                  0.66       0.66       0.52
// Where every tile has a CU, tagged values take another 3 to 15% off.  Scales
// with more 32 x 32 tiles than CUs take three iterations per chunk, whose
// registers let two tiles share a CU.  A scale that fits one workgroup needs no
// exchange at all (30x17: 0.15 against 0.20 ms, 20x15: 0.29 against 0.33).
static bool one_per_cu(const IterArgs& a, int centre)
{
    return (long long)cdiv((size_t)a.nx, (size_t)centre) * cdiv((size_t)a.ny, (size_t)centre) <= kSqOnePerCu;
}

static int launch_persist_square(const IterArgs& a, int nblocks, hipStream_t s)
{
    // the limit of the shape's own 4 iterations per chunk, whichever tile it takes
    if ((long long)a.max_iter / 4 + 1 >= kNbrMaxChunks) return OF_ERR_UNSUPPORTED;
    if (a.nx <= kSingleCols && a.ny <= kSingleCols) {
        const unsigned threads = 64 * cdiv((size_t)a.ny * kSingleCols, 64);
        hipLaunchKernelGGL(k_tvl1_single<4>, dim3(1), dim3(threads), 0, s, a);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            record_hip_error(e, "k_tvl1_single launch", __FILE__, __LINE__);
            return OF_ERR_HIP;
        }
        return OF_OK;
    }
    int st = OF_ERR_UNSUPPORTED;
    if (one_per_cu(a, 6)) st = launch_persist_tagged<16, 5>(a, nblocks, s);
    else if (one_per_cu(a, 14)) st = launch_persist_tagged<24, 5>(a, nblocks, s);
    else if (one_per_cu(a, 22)) st = launch_persist_tagged<32, 5>(a, nblocks, s);
    else if (one_per_cu(a, 24)) st = launch_persist_tagged<32, 4>(a, nblocks, s);
    if (st != OF_ERR_UNSUPPORTED) return st;
    // a flag counts the chunks of 4 iterations of any accepted limit, not those of 3
    if ((long long)a.max_iter / 3 + 1 >= kNbrMaxChunks) return launch_persist_sq<32, 4>(a, nblocks, s);
    return launch_persist_sq<32, 3>(a, nblocks, s);
}

int launch_persist(int K, int R, const IterArgs& a, int nblocks, hipStream_t s, int mode)
{
    if (mode != kPersistBarrier && mode != kPersistNeighbour) return OF_ERR_ARG;
    if (K == 4 && R == 0 && mode == kPersistNeighbour) return launch_persist_square(a, nblocks, s);
#define OF_PCASE(k, r)                                                            \
    if (K == k && R == r)                                                         \
        return mode == kPersistNeighbour ? launch_persist_kr<k, r, true>(a, nblocks, s) \
                                         : launch_persist_kr<k, r, false>(a, nblocks, s);
    if (K == 4 && R == 0) return launch_persist_kr<4, 0, false>(a, nblocks, s);
    OF_PCASE(1, 0) OF_PCASE(2, 0)
    OF_PCASE(1, 2) OF_PCASE(2, 2)
    OF_PCASE(1, 4) OF_PCASE(2, 4) OF_PCASE(4, 4)
    OF_PCASE(1, 8) OF_PCASE(2, 8) OF_PCASE(4, 8) OF_PCASE(8, 8)
#undef OF_PCASE
    return OF_ERR_UNSUPPORTED;
}

template <int K, int R>
static hipError_t launch_ls_kr(const LsPhase& ph, LsCtl* mc, unsigned grid,
                               unsigned long long* host_status, unsigned epoch, hipStream_t s)
{
    hipLaunchKernelGGL((k_ls_iter<K, R * 4 / kLsWaves, kLsWaves>), dim3(grid),
                       dim3(64 * kLsWaves), 0, s, ph, ph.pairs, mc, host_status, epoch);
    return hipGetLastError();
}

int launch_ls_iter(int K, int R, const LsPhase& ph, LsCtl* mc, unsigned grid,
                   unsigned long long* host_status, unsigned epoch, hipStream_t s)
{
    if (grid == 0 || ph.npairs < 1 || ph.npairs > kLsMaxPairs) return OF_ERR_ARG;
    hipError_t e = hipErrorInvalidValue;
#define OF_CASE(k, r) \
    if (K == k && R == r) e = launch_ls_kr<k, r>(ph, mc, grid, host_status, epoch, s);
    OF_CASE(1, 2) OF_CASE(2, 2)
    OF_CASE(1, 4) OF_CASE(2, 4) OF_CASE(4, 4)
    OF_CASE(1, 8) OF_CASE(2, 8) OF_CASE(4, 8) OF_CASE(8, 8)
#undef OF_CASE
    if (e != hipSuccess) {
        record_hip_error(e, "k_ls_iter launch", __FILE__, __LINE__);
        return OF_ERR_HIP;
    }
    return OF_OK;
}

template <int K, int R>
static int ls_resident_kr(unsigned* blocks)
{
    int dev = 0, per_cu = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, (const void*)k_ls_iter<K, R * 4 / kLsWaves, kLsWaves>, 64 * kLsWaves,
            0) != hipSuccess) {
        (void)hipGetLastError();
        return OF_ERR_HIP;
    }
    *blocks = (unsigned)std::max(1, per_cu) * (unsigned)std::max(1, cus);
    return OF_OK;
}

int ls_iter_resident(int K, int R, unsigned* blocks)
{
#define OF_CASE(k, r) \
    if (K == k && R == r) return ls_resident_kr<k, r>(blocks);
    OF_CASE(1, 2) OF_CASE(2, 2)
    OF_CASE(1, 4) OF_CASE(2, 4) OF_CASE(4, 4)
    OF_CASE(1, 8) OF_CASE(2, 8) OF_CASE(4, 8) OF_CASE(8, 8)
#undef OF_CASE
    return OF_ERR_ARG;
}

}  // namespace amdflow
