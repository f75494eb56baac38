// Ray-driven projector pair (semantics of radon_rd.c:15-189) for gfx950.
//
// Five sub-rays per detector bin (sub-ray i = 6b+1..6b+5 of bin b, radon_rd.c:123-185),
// each clipped to the square [-nh, nh]^2 and walked cell by cell; the length walked
// since the previous step is credited, with weight 1/5, to the cell just entered, and
// cells with row or column index 0 are skipped (radon_rd.c:44-66).  The walk repeats
// the reference build's arithmetic operation for operation (float geometry, double
// step parameters, double fused update rounded to float after every step).
//
// Forward: one thread per (bin, view) walks its five sub-rays in order.
// Back: one thread per pixel gathers, view by view and sub-ray by sub-ray in increasing
// index, the one step (if any) of each sub-ray's walk that enters the pixel, and applies
// it with the reference's rounding.  The walk is a merge of two increasing sequences of
// crossing parameters (x boundaries and y boundaries), so the step entering a cell, the
// step before it and whether the walk gets there follow from at most six of those
// parameters, computed exactly as the walk computes them.  Updates reach each pixel in
// the reference's own order: both projections are bit-identical to the reference's.
#include <algorithm>
#include <new>
#include <vector>

#include "epilogue.h"

namespace itomo {

static constexpr double kHalfPi = 3.141592653589793 / 2;

template <int ARITH>
__device__ __forceinline__ float rd_round(float v)
{
    if (ARITH == ITOMO_ARITH_FAST)  // gcc -ffast-math inline expansion of round()
        return truncf(__fadd_rn(v, copysignf(0.49999997f, v)));
    return (float)round((double)v);
}

// Entry/exit points of sub-ray i (radon_rd.c:123-179).
template <int ARITH>
__device__ __forceinline__ void rd_endpoints(int i, int npix, const RdView& g, float p1[2],
                                             float p2[2])
{
    const int nh = (int)(npix * 0.5);
    float t;
    if (ARITH == ITOMO_ARITH_FAST)
        t = (float)fabs(__fma_rn((double)i, 1.0 / 6.0, -(double)nh));
    else
        t = (float)fabs(__dsub_rn(__ddiv_rn((double)i, 6.0), (double)nh));
    const bool lt = g.lt_half_pi != 0;
    const bool gt = (double)g.theta > kHalfPi;
    if (i >= 3 * npix && lt) t = -t;
    if (i < 3 * npix && gt) t = -t;

    const float s = g.s, c = g.c;
    const float nhf = (float)nh, mnhf = (float)(-nh);
    float x1, y1, x2, y2;
    if (lt) {
        if (ARITH == ITOMO_ARITH_FAST) {
            y1 = __fmul_rn(__fadd_rn(t, __fmul_rn(mnhf, s)), g.rc);
            x1 = __fmul_rn(__fsub_rn(__fmul_rn(mnhf, c), t), g.rs);
            y2 = __fmul_rn(__fadd_rn(t, __fmul_rn(nhf, s)), g.rc);
            x2 = __fmul_rn(__fsub_rn(__fmul_rn(nhf, c), t), g.rs);
        } else {
            y1 = __fadd_rn(__fdiv_rn(__fmul_rn(mnhf, s), c), __fdiv_rn(t, c));
            x1 = __fsub_rn(__fdiv_rn(__fmul_rn(mnhf, c), s), __fdiv_rn(t, s));
            y2 = __fadd_rn(__fdiv_rn(__fmul_rn(nhf, s), c), __fdiv_rn(t, c));
            x2 = __fsub_rn(__fdiv_rn(__fmul_rn(nhf, c), s), __fdiv_rn(t, s));
        }
        if (y1 >= -nh && y1 <= nh) { p1[0] = mnhf; p1[1] = y1; }
        else                       { p1[0] = x1;   p1[1] = mnhf; }
        if (y2 >= -nh && y2 <= nh) { p2[0] = nhf;  p2[1] = y2; }
        else                       { p2[0] = x2;   p2[1] = nhf; }
    } else {
        if (ARITH == ITOMO_ARITH_FAST) {
            y1 = __fmul_rn(__fsub_rn(__fmul_rn(nhf, s), t), g.rc);
            x1 = __fmul_rn(__fadd_rn(t, __fmul_rn(mnhf, c)), g.rs);
            y2 = __fmul_rn(__fsub_rn(__fmul_rn(mnhf, s), t), g.rc);
            x2 = __fmul_rn(__fadd_rn(t, __fmul_rn(nhf, c)), g.rs);
        } else {
            y1 = __fsub_rn(__fdiv_rn(__fmul_rn(nhf, s), c), __fdiv_rn(t, c));
            x1 = __fadd_rn(__fdiv_rn(__fmul_rn(mnhf, c), s), __fdiv_rn(t, s));
            y2 = __fsub_rn(__fdiv_rn(__fmul_rn(mnhf, s), c), __fdiv_rn(t, c));
            x2 = __fadd_rn(__fdiv_rn(__fmul_rn(nhf, c), s), __fdiv_rn(t, s));
        }
        if (y1 >= -nh && y1 <= nh) { p1[0] = nhf;  p1[1] = y1; }
        else                       { p1[0] = x1;   p1[1] = mnhf; }
        if (y2 >= -nh && y2 <= nh) { p2[0] = mnhf; p2[1] = y2; }
        else                       { p2[0] = x2;   p2[1] = nhf; }
    }
}

// Float update of one pixel, exactly as the reference build rounds it.
template <int ARITH>
__device__ __forceinline__ float rd_back_update(float pix, float sv, float l)
{
    if (ARITH == ITOMO_ARITH_FAST)
        return (float)__fma_rn(__dmul_rn((double)sv, 0.2), (double)l, (double)pix);
    return (float)__dadd_rn((double)pix, __dmul_rn(__dmul_rn(0.2, (double)l), (double)sv));
}

template <int ARITH>
__device__ __forceinline__ float rd_fwd_update(float acc, float pix, float l)
{
    if (ARITH == ITOMO_ARITH_FAST)
        return (float)__fma_rn(__dmul_rn((double)l, 0.2), (double)pix, (double)acc);
    return (float)__dadd_rn((double)acc, __dmul_rn(__dmul_rn(0.2, (double)l), (double)pix));
}

// One sub-ray walk of the forward projection (radon_rd.c:15-71): returns the updated
// bin value.  The walk is capped at 4*npix+16 steps (a genuine walk takes at most
// 2*npix+2), so it always ends.
template <int ARITH, bool ONES>
__device__ float rd_walk(float acc, const float* __restrict__ img_in, int npix,
                         const float p1[2], const float p2[2])
{
    const int nh = (int)(npix * 0.5);
    const float d0 = __fsub_rn(p2[0], p1[0]), d1 = __fsub_rn(p2[1], p1[1]);
    // float sqrt via double: rounding a correctly rounded double square root to float
    // gives the correctly rounded float square root (53 >= 2*24 + 2).
    const float incr = (ARITH == ITOMO_ARITH_FAST)
                           ? (float)__dsqrt_rn((double)__fmaf_rn(d0, d0, __fmul_rn(d1, d1)))
                           : (float)__dsqrt_rn((double)__fadd_rn(__fmul_rn(d0, d0),
                                                                 __fmul_rn(d1, d1)));
    int ii = (int)rd_round<ARITH>(p1[0]);
    int jj = (int)rd_round<ARITH>(p1[1]);
    const float dx = (p2[0] > p1[0]) ? 1.0f : -1.0f;
    const float dy = (p2[1] > p1[1]) ? 1.0f : -1.0f;
    const double hx = 0.5 * (double)dx, hy = 0.5 * (double)dy;
    const double p1x = p1[0], p1y = p1[1], dd0 = d0, dd1 = d1;
    float alpha = 0.0f, alpha_old = 0.0f;
    float ax = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)ii, hx), p1x), dd0);
    float ay = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)jj, hy), p1y), dd1);
    const int cap = 4 * npix + 16;
    bool pend = false;  // an update (pv, pl) waits for the next step
    float pv = 0.0f, pl = 0.0f;
    for (int step = 0; alpha <= 1.0f && step < cap; ++step) {
        if (ax < ay) {
            alpha = ax;
            ii = (int)__fadd_rn((float)ii, dx);
            ax = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)ii, hx), p1x), dd0);
        } else if (ax > ay) {
            alpha = ay;
            jj = (int)__fadd_rn((float)jj, dy);
            ay = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)jj, hy), p1y), dd1);
        } else if (ax == ay) {
            alpha = ay;
            ii = (int)__fadd_rn((float)ii, dx);
            jj = (int)__fadd_rn((float)jj, dy);
            ax = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)ii, hx), p1x), dd0);
            ay = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)jj, hy), p1y), dd1);
        } else {
            break;  // NaN step parameter: the reference would never terminate
        }
        const float l = __fmul_rn(__fsub_rn(alpha, alpha_old), incr);
        const int i = ii + nh, j = jj + nh;
        const bool in = i > 0 && i < npix && j > 0 && j < npix;
        // this step's pixel is loaded now and added one step later, so the load is in
        // flight while the walk computes the next step; the updates keep their order
        const float v = (in && !ONES) ? img_in[(int64_t)i * npix + j] : 1.0f;
        if (pend) acc = rd_fwd_update<ARITH>(acc, pv, pl);
        pend = in;
        pv = v;
        pl = l;
        alpha_old = alpha;
    }
    if (pend) acc = rd_fwd_update<ARITH>(acc, pv, pl);
    return acc;
}

// Whether a bin's forward words index the transposed image.  After equally many steps the walks
// that start on the square's x edges are in the same image row, in neighbouring columns, and
// those that start on its y edges in the same column: the latter read the transposed copy, so
// that the lanes of a wave (64 neighbouring bins) gather from neighbouring addresses.  (Chosen
// per view, by the steeper axis, and with the sub-rays of a list unaligned, a wave's gather
// touches up to 64 lines: 256^2 x 304 views, 263 us a call against 158.)
template <int ARITH>
__device__ __forceinline__ bool rd_fwd_transposed(const RdView& g, int b, int npix)
{
    float p1[2], p2[2];
    rd_endpoints<ARITH>(6 * b + 3, npix, g, p1, p2);
    return fabsf(p1[0]) != (float)(int)(npix * 0.5);
}

// The cached system matrix of a plan (see rd_matrix_ensure), or all null.
struct RdMat {
    const unsigned* ent;
    const int64_t* off;
};

// A matrix word: two bits of code, 30 of payload.  A credited length l is a float in [0, 2),
// whose two top bits are zero (the recording counts any that is not, and the matrix is then
// declined), so a step and its length fit 32 bits without loss.
//   forward: codes 0, 1, 2 move the image index by a, b, a + b (RdSteps) and credit l there;
//   back:    codes 0, 1 move the sinogram index by 0, 1 and credit l from there, code 2 sets
//            it and adds the bin plainly (row-sum and column-sum views);
//   both:    code 3 sets the index and credits nothing (starts, and the padding).
constexpr unsigned kRdPayload = 0x3fffffffu;
constexpr int kRdBatch = 16;               // words of a lane handled together, four 16-byte loads
constexpr int kRdRing = 4;                 // batches in registers; lists are padded to a ring
constexpr int kRdPad = kRdBatch * kRdRing;

// The index steps of a bin's forward words: (row, column) moves along the view's usual walk.
struct RdSteps {
    int a, b;
};

__device__ __forceinline__ RdSteps rd_fwd_steps(const RdView& g, int npix, bool transposed)
{
    const int si = transposed ? 1 : npix, sj = transposed ? npix : 1;
    return {g.lt_half_pi ? si : -si, sj};
}

// Replays one output's words (nb batches of them, a multiple of kRdRing) into acc, in order.
// What bounds it is the stream of words: it is read once per call, and there are only about as
// many waves as SIMDs (a bin or a pixel is one serial chain of rounded updates), so each wave
// keeps three batches of its lanes' words in flight (12 KB) and the gathers of one batch while
// it updates the one before.  No load is predicated: batches past the end repeat the last one
// and the padding gathers index 0.
template <int ARITH, bool ONES, bool BACK>
__device__ __forceinline__ float rd_replay(float acc, const uint4* __restrict__ e, int nb,
                                           const float* __restrict__ src, unsigned last,
                                           RdSteps st)
{
    if (nb <= 0) return acc;
    unsigned q[kRdRing][kRdBatch];
    float v[2][kRdBatch];
    unsigned idx = 0;
    const int ab = st.a + st.b;
    auto load = [&](unsigned (&d)[kRdBatch], int batch) {
        const uint4* p = e + (int64_t)min(batch, nb - 1) * (kRdBatch / 4 * 64);
#pragma unroll
        for (int g = 0; g < kRdBatch / 4; ++g) {
            const uint4 w = p[g * 64];
            d[4 * g] = w.x;
            d[4 * g + 1] = w.y;
            d[4 * g + 2] = w.z;
            d[4 * g + 3] = w.w;
        }
    };
    auto gather = [&](const unsigned (&d)[kRdBatch], float (&x)[kRdBatch]) {
#pragma unroll
        for (int u = 0; u < kRdBatch; ++u) {
            const unsigned w = d[u], pay = w & kRdPayload;
            if (BACK) {
                idx = w >= 0x80000000u ? pay : idx + (w >> 30);
                x[u] = ONES ? 1.0f : src[idx];
            } else {
                const int step = w >= 0x80000000u ? ab : (w & 0x40000000u) ? st.b : st.a;
                idx = w >= 0xc0000000u ? pay : idx + (unsigned)step;
                x[u] = ONES ? 1.0f : src[min(idx, last)];   // a start may lie one step outside
            }
        }
    };
    auto update = [&](const unsigned (&d)[kRdBatch], const float (&x)[kRdBatch]) {
#pragma unroll
        for (int u = 0; u < kRdBatch; ++u) {
            const float l = __uint_as_float(d[u] & kRdPayload);
            float n;
            if (BACK)
                n = d[u] >= 0x80000000u ? __fadd_rn(acc, x[u]) : rd_back_update<ARITH>(acc, x[u], l);
            else
                n = rd_fwd_update<ARITH>(acc, x[u], l);
            acc = d[u] >= 0xc0000000u ? acc : n;
        }
    };
#pragma unroll
    for (int r = 0; r < kRdRing - 1; ++r) load(q[r], r);
#pragma unroll
    for (int u = 0; u < kRdBatch; ++u) {
        q[kRdRing - 1][u] = 0xc0000000u;
        v[1][u] = 0.0f;
    }
#pragma unroll 1
    for (int j = 0; j < nb; j += kRdRing) {
#pragma unroll
        for (int r = 0; r < kRdRing; ++r) {
            constexpr int kPrev = kRdRing - 1;
            gather(q[r], v[r & 1]);
            __builtin_amdgcn_sched_barrier(0);
            update(q[(r + kPrev) % kRdRing], v[(r & 1) ^ 1]);
            load(q[(r + kPrev) % kRdRing], j + r + kPrev);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    update(q[kRdRing - 1], v[(kRdRing - 1) & 1]);
    return acc;
}

template <int ARITH, int EPI, bool ONES>
__global__ void __launch_bounds__(64)
rd_fwd_kernel(const RdView* __restrict__ geom, int npix, const float* __restrict__ image,
              const float* __restrict__ imageT, float* __restrict__ out, int64_t img_stride,
              int64_t sino_stride, int accumulate, EpiArgs e, RdMat mat)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = b < npix;
    const int v = blockIdx.y, z = blockIdx.z;
    const RdView g = geom[v];
    image += (int64_t)z * img_stride;
    const int64_t soff = (int64_t)z * sino_stride;
    const int64_t o = (int64_t)v * npix + b;
    double p0 = 0.0;
    if (active) {
        float acc = (EPI == EPI_STORE && accumulate) ? out[soff + o] : 0.0f;
        const float* imgT = imageT + (int64_t)z * img_stride;
        if (mat.ent && g.kind == RD_RAYS) {
            // the bin's cached updates, in order (bitwise the walk's), from the image or its
            // transpose as they were recorded
            const int64_t chunk = (int64_t)v * gridDim.x + blockIdx.x;
            const int64_t off = mat.off[chunk];
            const bool t = rd_fwd_transposed<ARITH>(g, b, npix);
            acc = rd_replay<ARITH, ONES, false>(
                acc, (const uint4*)(mat.ent + off) + threadIdx.x,
                (int)((mat.off[chunk + 1] - off) / (64 * kRdBatch)),
                t ? imgT : image, (unsigned)(npix * npix - 1), rd_fwd_steps(g, npix, t));
        } else if (mat.ent && g.kind == RD_ROWSUM && !ONES) {
#pragma unroll 8
            for (int j = 0; j < npix; ++j) acc = __fadd_rn(acc, imgT[(int64_t)j * npix + b]);
        } else if (g.kind == RD_COLSUM) {
            const int i = npix - 1 - b;  // bin N-1-i <- column i, i >= 1
            if (i >= 1)
                for (int j = 0; j < npix; ++j)
                    acc = __fadd_rn(acc, ONES ? 1.0f : image[(int64_t)j * npix + i]);
        } else if (g.kind == RD_ROWSUM) {
            for (int j = 0; j < npix; ++j)
                acc = __fadd_rn(acc, ONES ? 1.0f : image[(int64_t)b * npix + j]);
        } else {
            for (int k = 1; k <= 5; ++k) {
                float p1[2], p2[2];
                rd_endpoints<ARITH>(6 * b + k, npix, g, p1, p2);
                acc = rd_walk<ARITH, ONES>(acc, image, npix, p1, p2);
            }
        }
        out[soff + o] = epi_forward<EPI>(acc, o, soff, z, e, &p0);
    }
    if (epi_has_partials(EPI) && e.partials) {
        const int blk = blockIdx.y * gridDim.x + blockIdx.x;
        block_partials3(p0, 0.0, 0.0,
                        e.partials + ((int64_t)z * e.blocks_per_slice + blk) * 3);
    }
}

// Crossing parameter of the walk's m-th boundary along one axis: the boundary between
// cells c0 + m*dc and c0 + (m+1)*dc, as the walk computes it (radon_rd.c:31-32).
__device__ __forceinline__ float rd_cross(int c0, int m, int dc, double h, float p, float d)
{
    return (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)(c0 + m * dc), h), (double)p),
                            (double)d);
}

// The step of one sub-ray's walk that enters cell (ii, jj), if the walk takes it:
// returns true and the credited length l.  The walk merges the x crossings X(0) < X(1)
// < ... with the y crossings Y(0) < Y(1) < ... (equal values make one diagonal step);
// x reaches ii after X(sx-1) and leaves it at X(sx), likewise for y, so the cell is
// entered at E = max(X(sx-1), Y(sy-1)) if E precedes both X(sx) and Y(sy).  The step
// before is the larger of the crossings preceding E; the walk takes the step while the
// one before it is <= 1 (radon_rd.c:28), and credits (E - previous) * |p2 - p1|.
template <int ARITH>
__device__ __forceinline__ bool rd_cell_step(const float p1[2], const float p2[2], int ii, int jj,
                                             float* l_out)
{
    const float d0 = __fsub_rn(p2[0], p1[0]), d1 = __fsub_rn(p2[1], p1[1]);
    const int i0 = (int)rd_round<ARITH>(p1[0]);
    const int j0 = (int)rd_round<ARITH>(p1[1]);
    const int dx = (p2[0] > p1[0]) ? 1 : -1, dy = (p2[1] > p1[1]) ? 1 : -1;
    const int sx = (ii - i0) * dx, sy = (jj - j0) * dy;
    if (sx < 0 || sy < 0 || (sx == 0 && sy == 0)) return false;  // behind, or the start cell
    const double hx = 0.5 * (double)dx, hy = 0.5 * (double)dy;
    const float ninf = __int_as_float(0xff800000);
    const float Ex = sx > 0 ? rd_cross(i0, sx - 1, dx, hx, p1[0], d0) : ninf;
    const float Ey = sy > 0 ? rd_cross(j0, sy - 1, dy, hy, p1[1], d1) : ninf;
    const float E = fmaxf(Ex, Ey);
    if (!(E < rd_cross(i0, sx, dx, hx, p1[0], d0))) return false;
    if (!(E < rd_cross(j0, sy, dy, hy, p1[1], d1))) return false;
    const float Xp = (Ex >= Ey && sx >= 2) ? rd_cross(i0, sx - 2, dx, hx, p1[0], d0) : ninf;
    const float Yp = (Ey >= Ex && sy >= 2) ? rd_cross(j0, sy - 2, dy, hy, p1[1], d1) : ninf;
    const float prev = Ex > Ey ? fmaxf(Xp, Ey) : (Ey > Ex ? fmaxf(Yp, Ex) : fmaxf(Xp, Yp));
    const float aold = (prev == ninf) ? 0.0f : prev;
    if (!(aold <= 1.0f)) return false;
    const float incr = (ARITH == ITOMO_ARITH_FAST)
                           ? (float)__dsqrt_rn((double)__fmaf_rn(d0, d0, __fmul_rn(d1, d1)))
                           : (float)__dsqrt_rn((double)__fadd_rn(__fmul_rn(d0, d0),
                                                                 __fmul_rn(d1, d1)));
    *l_out = __fmul_rn(__fsub_rn(E, aold), incr);
    return true;
}

// Back projection as a gather: one thread per pixel (16 x 16 per block), all views in
// order.  Sub-ray i lies on the line y*c - x*s = tau(i) with tau(i) = nh - i/6, except,
// for odd npix, sub-rays 6nh+1 and 6nh+2, whose t >= 0 below 3*npix keeps its sign
// (radon_rd.c:125-128) and puts them on tau = i/6 - nh.  A pixel's cell meets the lines
// with |tau - tau_c| <= (|c| + |s|)/2, tau_c = jj*c - ii*s; the candidates are those
// sub-rays plus one more on each side (a sixth of a pixel, far above the walk's
// rounding), and rd_cell_step decides each exactly.
template <int ARITH, bool ONES>
__global__ void __launch_bounds__(256)
rd_back_gather_kernel(const RdView* __restrict__ geom, int nang, int npix,
                      const float* __restrict__ sino, float* __restrict__ image,
                      int64_t sino_stride, int64_t img_stride, int accumulate)
{
    const int cc = blockIdx.x * 16 + (threadIdx.x & 15);  // image column (y cell)
    const int r = blockIdx.y * 16 + (threadIdx.x >> 4);   // image row (x cell)
    if (r >= npix || cc >= npix) return;
    image += (int64_t)blockIdx.z * img_stride;
    sino += (int64_t)blockIdx.z * sino_stride;
    const int64_t o = (int64_t)r * npix + cc;
    float pix = accumulate ? image[o] : 0.0f;
    const int nh = (int)(npix * 0.5);
    const int ii = r - nh, jj = cc - nh;
    const bool inner = r >= 1 && cc >= 1;
    for (int v = 0; v < nang; ++v) {
        const RdView g = geom[v];
        const float* row = sino + (int64_t)v * npix;
        if (g.kind == RD_COLSUM) {
            if (cc >= 1) pix = __fadd_rn(pix, ONES ? 1.0f : row[npix - 1 - cc]);
        } else if (g.kind == RD_ROWSUM) {
            pix = __fadd_rn(pix, ONES ? 1.0f : row[r]);
        } else if (inner) {
            const double sd = (double)g.s, cd = (double)g.c;
            const double tc = (double)jj * cd - (double)ii * sd;
            const double hw = 0.5 * (fabs(cd) + fabs(sd));
            int ilo = (int)floor(6.0 * ((double)nh - tc - hw)) - 1;
            int ihi = (int)ceil(6.0 * ((double)nh - tc + hw)) + 1;
            if ((npix & 1) && tc - hw - 1.0 / 3.0 <= 2.0 / 6.0 && tc + hw + 1.0 / 3.0 >= 1.0 / 6.0) {
                ilo = min(ilo, 6 * nh + 1);
                ihi = max(ihi, 6 * nh + 2);
            }
            ilo = max(ilo, 1);
            ihi = min(ihi, 6 * npix - 1);
            for (int i = ilo; i <= ihi; ++i) {
                if (i % 6 == 0) continue;
                float p1[2], p2[2], l;
                rd_endpoints<ARITH>(i, npix, g, p1, p2);
                if (!rd_cell_step<ARITH>(p1, p2, ii, jj, &l)) continue;
                pix = rd_back_update<ARITH>(pix, ONES ? 1.0f : row[i / 6], l);
            }
        }
    }
    image[o] = pix;
}

// ---- the cached system matrix ------------------------------------------------------
//
// With 288 GB of HBM per GPU the exact system matrix of a small ray-driven geometry fits
// many times over (4 bytes per walk step, once per direction), and replaying it turns
// both projections into streaming passes instead of latency-bound walks.  The words are what
// the walks compute: per bin the steps of its five sub-rays that enter an image cell, in walk
// order (indices into the image or its transpose, rd_fwd_transposed); per
// pixel, in view order, the row-sum and column-sum views' bins and every sub-ray step entering
// it.  Replaying them in that order with the same update arithmetic gives the walks' results
// bit for bit.
// Word n of lane k of a 64-output chunk lies at off[chunk] + 256 (n/4) + 4 k + n%4.
// Against eight-byte {index, length} entries loaded in predicated batches, us per call forward
// and back: 64^2 x 45 views 76 -> 31 and 39 -> 24, 256^2 x 304 404 -> 158 and 295 -> 146 (3.6
// and 4.3 TB/s of words), two slices of it 826 -> 262 and 367 -> 280.

// Writes (FILL) or counts an output's words.
template <bool FILL>
struct RdWords {
    unsigned* out;
    int n = 0;
    unsigned bad = 0;

    __device__ __forceinline__ void put(unsigned code, unsigned payload)
    {
        if (FILL) out[(n >> 2) * 256 + (n & 3)] = code << 30 | payload;
        ++n;
    }
    __device__ __forceinline__ void credit(unsigned code, float l)
    {
        const unsigned u = __float_as_uint(l);
        bad |= u & ~kRdPayload;
        put(code, u & kRdPayload);
    }
    __device__ __forceinline__ void pad(int words)
    {
        if (FILL)
            while (n < words) put(3, 0);
        n = words;
    }
    // The number of words, or -1 when a length does not fit.
    __device__ __forceinline__ int count() const { return bad ? -1 : n; }
};

// One sub-ray walk of radon_rd.c:15-71 (the steps of rd_walk) recording the steps that
// enter an image cell.
template <int ARITH, bool FILL>
__device__ void rd_walk_record(int npix, const float p1[2], const float p2[2],
                               RdWords<FILL>& words, RdSteps st, bool transposed)
{
    const int nh = (int)(npix * 0.5);
    const float d0 = __fsub_rn(p2[0], p1[0]), d1 = __fsub_rn(p2[1], p1[1]);
    const float incr = (ARITH == ITOMO_ARITH_FAST)
                           ? (float)__dsqrt_rn((double)__fmaf_rn(d0, d0, __fmul_rn(d1, d1)))
                           : (float)__dsqrt_rn((double)__fadd_rn(__fmul_rn(d0, d0),
                                                                 __fmul_rn(d1, d1)));
    int ii = (int)rd_round<ARITH>(p1[0]);
    int jj = (int)rd_round<ARITH>(p1[1]);
    const float dx = (p2[0] > p1[0]) ? 1.0f : -1.0f;
    const float dy = (p2[1] > p1[1]) ? 1.0f : -1.0f;
    const double hx = 0.5 * (double)dx, hy = 0.5 * (double)dy;
    const double p1x = p1[0], p1y = p1[1], dd0 = d0, dd1 = d1;
    float alpha = 0.0f, alpha_old = 0.0f;
    float ax = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)ii, hx), p1x), dd0);
    float ay = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)jj, hy), p1y), dd1);
    const int cap = 4 * npix + 16;
    const int mi = (int)dx * (transposed ? 1 : npix), mj = (int)dy * (transposed ? npix : 1);
    bool live = false;   // the step before was recorded
    for (int step = 0; alpha <= 1.0f && step < cap; ++step) {
        int move;
        if (ax < ay) {
            move = mi;
            alpha = ax;
            ii = (int)__fadd_rn((float)ii, dx);
            ax = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)ii, hx), p1x), dd0);
        } else if (ax > ay) {
            move = mj;
            alpha = ay;
            jj = (int)__fadd_rn((float)jj, dy);
            ay = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)jj, hy), p1y), dd1);
        } else if (ax == ay) {
            move = mi + mj;
            alpha = ay;
            ii = (int)__fadd_rn((float)ii, dx);
            jj = (int)__fadd_rn((float)jj, dy);
            ax = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)ii, hx), p1x), dd0);
            ay = (float)__ddiv_rn(__dsub_rn(__dadd_rn((double)jj, hy), p1y), dd1);
        } else {
            break;
        }
        const float l = __fmul_rn(__fsub_rn(alpha, alpha_old), incr);
        const int i = ii + nh, jc = jj + nh;
        if (i > 0 && i < npix && jc > 0 && jc < npix) {
            const int index = transposed ? jc * npix + i : i * npix + jc;
            const int code = move == st.a ? 0 : move == st.b ? 1 : move == st.a + st.b ? 2 : -1;
            // the cell before lies at most one step outside the image, so its index is >= 0
            if (code < 0 || !live) words.put(3, (unsigned)(index - (code < 0 ? st.a : move)));
            words.credit(code < 0 ? 0 : code, l);
            live = true;
        } else {
            live = false;
        }
        alpha_old = alpha;
    }
}

// Forward rows: one thread per (bin, view), as rd_fwd_kernel: the five sub-rays' steps (a sum
// view has none: its bins add image rows or columns).
template <int ARITH, bool FILL>
__global__ void __launch_bounds__(64)
rd_fwd_record_kernel(const RdView* __restrict__ geom, int npix, int* __restrict__ cnt,
                     unsigned* __restrict__ ent, const int64_t* __restrict__ off)
{
    const int b = blockIdx.x * 64 + threadIdx.x;
    const int v = blockIdx.y;
    const RdView g = geom[v];
    const int64_t chunk = (int64_t)v * gridDim.x + blockIdx.x;
    RdWords<FILL> words{FILL ? ent + off[chunk] + 4 * threadIdx.x : nullptr};
    if (g.kind == RD_RAYS) {
        const bool t = rd_fwd_transposed<ARITH>(g, b, npix);
        for (int k = 1; k <= 5; ++k) {
            if (b < npix) {
                float p1[2], p2[2];
                rd_endpoints<ARITH>(6 * b + k, npix, g, p1, p2);
                rd_walk_record<ARITH, FILL>(npix, p1, p2, words, rd_fwd_steps(g, npix, t), t);
            }
            // the chunk's bins begin their next sub-ray together, as near to each other as they
            // began the first: a chunk is then as long as its longest sub-rays one after
            // another, not as its longest list (256^2 x 304: 0.01% more words; the call 157 us
            // instead of 234)
            int m = words.n;
            for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
            words.pad(m);
        }
    }
    if (FILL)
        words.pad((int)((off[chunk + 1] - off[chunk]) / 64));
    else if (b < npix)
        cnt[(int64_t)v * npix + b] = words.count();
}

// Back columns: one thread per pixel, the candidates of rd_back_gather_kernel.
template <int ARITH, bool FILL>
__global__ void __launch_bounds__(256)
rd_back_record_kernel(const RdView* __restrict__ geom, int nang, int npix,
                      int* __restrict__ cnt, unsigned* __restrict__ ent,
                      const int64_t* __restrict__ off)
{
    const int cc = blockIdx.x * 16 + (threadIdx.x & 15);
    const int r = blockIdx.y * 16 + (threadIdx.x >> 4);
    if (r >= npix || cc >= npix) return;
    const int64_t o = (int64_t)r * npix + cc;
    RdWords<FILL> words{FILL ? ent + off[o >> 6] + 4 * (o & 63) : nullptr};
    const int nh = (int)(npix * 0.5);
    const int ii = r - nh, jj = cc - nh;
    const bool inner = r >= 1 && cc >= 1;
    int last = -2;
    for (int v = 0; v < nang; ++v) {
        const RdView g = geom[v];
        const int rowbase = v * npix;
        if (g.kind == RD_COLSUM) {
            if (cc >= 1) words.put(2, (unsigned)(last = rowbase + npix - 1 - cc));
        } else if (g.kind == RD_ROWSUM) {
            words.put(2, (unsigned)(last = rowbase + r));
        } else if (inner) {
            const double sd = (double)g.s, cd = (double)g.c;
            const double tc = (double)jj * cd - (double)ii * sd;
            const double hw = 0.5 * (fabs(cd) + fabs(sd));
            int ilo = (int)floor(6.0 * ((double)nh - tc - hw)) - 1;
            int ihi = (int)ceil(6.0 * ((double)nh - tc + hw)) + 1;
            if ((npix & 1) && tc - hw - 1.0 / 3.0 <= 2.0 / 6.0 && tc + hw + 1.0 / 3.0 >= 1.0 / 6.0) {
                ilo = min(ilo, 6 * nh + 1);
                ihi = max(ihi, 6 * nh + 2);
            }
            ilo = max(ilo, 1);
            ihi = min(ihi, 6 * npix - 1);
            for (int i = ilo; i <= ihi; ++i) {
                if (i % 6 == 0) continue;
                float p1[2], p2[2], l;
                rd_endpoints<ARITH>(i, npix, g, p1, p2);
                if (!rd_cell_step<ARITH>(p1, p2, ii, jj, &l)) continue;
                const int bin = rowbase + i / 6, d = bin - last;
                const bool near = d == 0 || d == 1;
                if (!near) words.put(3, (unsigned)bin);
                words.credit(near ? d : 0, l);
                last = bin;
            }
        }
    }
    if (FILL)
        words.pad((int)((off[(o >> 6) + 1] - off[o >> 6]) / 64));
    else
        cnt[o] = words.count();
}

// Back projection from the cached columns: one thread per pixel, updates in view order
// with rd_back_gather_kernel's arithmetic.
template <int ARITH, bool ONES>
__global__ void __launch_bounds__(64)
rd_back_matrix_kernel(const unsigned* __restrict__ ent, const int64_t* __restrict__ off,
                      int npix, const float* __restrict__ sino, float* __restrict__ image,
                      int64_t sino_stride, int64_t img_stride, int accumulate)
{
    const int64_t o = (int64_t)blockIdx.x * 64 + threadIdx.x;
    if (o >= (int64_t)npix * npix) return;
    image += (int64_t)blockIdx.y * img_stride;
    sino += (int64_t)blockIdx.y * sino_stride;
    const float pix = accumulate ? image[o] : 0.0f;
    const int64_t base = off[blockIdx.x];
    image[o] = rd_replay<ARITH, ONES, true>(
        pix, (const uint4*)(ent + base) + threadIdx.x,
        (int)((off[blockIdx.x + 1] - base) / (64 * kRdBatch)), sino, 0, RdSteps{0, 1});
}

namespace {

// Chunk offsets of a matrix from its per-output word counts: outputs are grouped 64 at a time
// within rows of `row` outputs, and a chunk holds 64 x (its largest count, padded) words; the
// last offset is the total.  False when an output could not be recorded (a count below 0).
bool chunk_layout(const std::vector<int>& cnt, int64_t nout, int64_t chunks_per_row,
                  int64_t row, std::vector<int64_t>* off)
{
    const int64_t nrows = nout / row;
    off->assign((size_t)(nrows * chunks_per_row + 1), 0);
    int64_t total = 0;
    for (int64_t rr = 0; rr < nrows; ++rr)
        for (int64_t c = 0; c < chunks_per_row; ++c) {
            int64_t m = 0;
            for (int64_t k = c * 64; k < std::min<int64_t>(row, c * 64 + 64); ++k) {
                if (cnt[(size_t)(rr * row + k)] < 0) return false;
                m = std::max<int64_t>(m, cnt[(size_t)(rr * row + k)]);
            }
            total += (m + kRdPad - 1) / kRdPad * kRdPad * 64;
            (*off)[(size_t)(rr * chunks_per_row + c) + 1] = total;
        }
    return true;
}

}  // namespace

void rd_matrix_free(const Plan& p)
{
    void* ptrs[] = {p.rdf_ent, p.rdf_off, p.rdb_ent, p.rdb_off};
    for (void* q : ptrs)
        if (q) (void)hipFree(q);
    p.rdf_ent = p.rdb_ent = nullptr;
    p.rdf_off = p.rdb_off = nullptr;
    p.rd_mat_bytes = 0;
}

// hipMalloc that, when the device is out of memory, leaves no error behind: the matrix is
// then declined and the walks stay in use.
template <typename T>
static bool try_alloc(T** ptr, size_t bytes)
{
    if (hipMalloc((void**)ptr, bytes) == hipSuccess) return true;
    (void)hipGetLastError();
    *ptr = nullptr;
    return false;
}

// The matrix of p, on st; returns ITOMO_OK with rd_mat_state unchanged when it is declined.
template <int ARITH>
static int rd_matrix_build(const Plan& p, int* cntf, int* cntb, hipStream_t st)
{
    const int n = p.npix, V = p.nang;
    const int64_t n2 = (int64_t)n * n, nf = (int64_t)V * n;
    const int fcpr = (n + 63) / 64;                       // forward chunks per view
    const RdView* g = (const RdView*)p.d_geom;
    int rc;
    rd_fwd_record_kernel<ARITH, false><<<dim3(fcpr, V), 64, 0, st>>>(g, n, cntf, nullptr,
                                                                       nullptr);
    rd_back_record_kernel<ARITH, false><<<dim3((n + 15) / 16, (n + 15) / 16), 256, 0, st>>>(
        g, V, n, cntb, nullptr, nullptr);
    rc = check_hip(hipGetLastError(), "rd matrix: count launch");
    std::vector<int64_t> of, ob;
    std::vector<int> cf((size_t)nf), cb((size_t)n2);
    if (!rc) rc = check_hip(hipMemcpyAsync(cf.data(), cntf, nf * sizeof(int),
                                           hipMemcpyDeviceToHost, st), "rd matrix: counts");
    if (!rc) rc = check_hip(hipMemcpyAsync(cb.data(), cntb, n2 * sizeof(int),
                                           hipMemcpyDeviceToHost, st), "rd matrix: counts");
    if (!rc) rc = check_hip(hipStreamSynchronize(st), "rd matrix: sync");
    if (rc) return rc;
    // back: pixels in row-major chunks of 64 (one "row" of all n2 outputs)
    if (!chunk_layout(cf, nf, fcpr, n, &of) || !chunk_layout(cb, n2, (n2 + 63) / 64, n2, &ob))
        return ITOMO_OK;
    const int64_t tf = of.back(), tb = ob.back();
    const size_t bytes = (size_t)(tf + tb) * sizeof(unsigned);
    if (bytes > kRdMatrixMaxBytes) return ITOMO_OK;
    if (!try_alloc(&p.rdf_ent, std::max<int64_t>(tf, 4) * sizeof(unsigned)) ||
        !try_alloc(&p.rdb_ent, std::max<int64_t>(tb, 4) * sizeof(unsigned)) ||
        !try_alloc(&p.rdf_off, of.size() * sizeof(int64_t)) ||
        !try_alloc(&p.rdb_off, ob.size() * sizeof(int64_t)))
        return ITOMO_OK;
    rc = check_hip(hipMemcpy(p.rdf_off, of.data(), of.size() * sizeof(int64_t),
                             hipMemcpyHostToDevice), "rd matrix");
    if (!rc) rc = check_hip(hipMemcpy(p.rdb_off, ob.data(), ob.size() * sizeof(int64_t),
                                      hipMemcpyHostToDevice), "rd matrix");
    if (rc) return rc;
    rd_fwd_record_kernel<ARITH, true><<<dim3(fcpr, V), 64, 0, st>>>(g, n, nullptr, p.rdf_ent,
                                                                      p.rdf_off);
    rd_back_record_kernel<ARITH, true><<<dim3((n + 15) / 16, (n + 15) / 16), 256, 0, st>>>(
        g, V, n, nullptr, p.rdb_ent, p.rdb_off);
    rc = check_hip(hipGetLastError(), "rd matrix: fill launch");
    if (!rc) rc = check_hip(hipStreamSynchronize(st), "rd matrix: sync");
    if (rc) return rc;
    p.rd_mat_bytes = bytes;
    p.rd_mat_state = 1;
    return ITOMO_OK;
}

// A launch recorded into a stream capture keeps the matrix's addresses in the graph: from
// then on the matrix stays until the plan is destroyed (itomo_plan_rd_matrix refuses to
// drop it).
void rd_matrix_note_use(const Plan& p, hipStream_t st)
{
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) == hipSuccess && cs != hipStreamCaptureStatusNone)
        p.rd_mat_pinned = 1;
}

int rd_matrix_ensure(const Plan& p, hipStream_t st)
{
    if (p.projector != ITOMO_PROJ_RD || p.rd_mat_state != 0 || scratch_region_active())
        return ITOMO_OK;
    // no synchronising build under stream capture: the walks are captured instead
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    int rc = check_hip(hipStreamIsCapturing(st, &cs), "rd matrix: capture status");
    if (rc || cs != hipStreamCaptureStatusNone) return rc;
    p.rd_mat_state = -1;
    // upper bound of the words (a walk takes at most 2 npix + 2 steps): skip the counting
    // passes when even a fraction of it cannot fit
    const double bound = 8.0 * 5.0 * p.nang * (double)p.npix * (1.5 * p.npix);
    if (bound > 4.0 * (double)kRdMatrixMaxBytes) return ITOMO_OK;
    // the words hold 30-bit indices, of starts up to a row outside the image
    const int64_t nf = (int64_t)p.nang * p.npix, n2 = (int64_t)p.npix * p.npix;
    if (nf > kRdPayload || n2 + p.npix > kRdPayload) return ITOMO_OK;
    rc = check_hip(hipStreamSynchronize(st), "rd matrix: sync");
    if (rc) return rc;
    int *cntf = nullptr, *cntb = nullptr;
    if (try_alloc(&cntf, nf * sizeof(int)) && try_alloc(&cntb, n2 * sizeof(int))) {
        try {
            rc = p.arith == ITOMO_ARITH_FAST
                     ? rd_matrix_build<ITOMO_ARITH_FAST>(p, cntf, cntb, st)
                     : rd_matrix_build<ITOMO_ARITH_IEEE>(p, cntf, cntb, st);
        } catch (const std::bad_alloc&) {   // no host memory for the counts: declined
        }
    }
    (void)hipFree(cntf);
    (void)hipFree(cntb);
    if (p.rd_mat_state != 1) rd_matrix_free(p);
    return rc;
}

namespace {

template <int ARITH, int EPI, bool ONES>
int launch_rd_fwd(const Plan& p, const float* image, float* out, int nslices,
                  int accumulate, const EpiArgs& e, hipStream_t st)
{
    dim3 block(64), grid((p.npix + 63) / 64, p.nang, nslices);
    const float* imageT = image;
    if (p.rd_mat_state == 1) {
        rd_matrix_note_use(p, st);
        if (!ONES) {   // the transposed copy the recorded entries of some views index
            Scratch s;
            int rc = get_scratch(p, nslices, &s, st);
            if (!rc) rc = launch_transpose(image, s.xT, p.npix, nslices, st);
            if (rc) return rc;
            imageT = s.xT;
        }
    }
    const RdMat mat = p.rd_mat_state == 1
                          ? RdMat{p.rdf_ent, p.rdf_off}
                          : RdMat{nullptr, nullptr};
    rd_fwd_kernel<ARITH, EPI, ONES><<<grid, block, 0, st>>>(
        (const RdView*)p.d_geom, p.npix, image, imageT, out, (int64_t)p.npix * p.npix,
        (int64_t)p.nang * p.npix, accumulate, e, mat);
    return ITOMO_OK;
}

template <int ARITH>
int dispatch_rd_fwd(const Plan& p, int epi, int ones, const float* image, float* out,
                    int nslices, int accumulate, const EpiArgs& e, hipStream_t st)
{
    switch (epi) {
    case EPI_STORE:
        if (ones) return launch_rd_fwd<ARITH, EPI_STORE, true>(p, image, out, nslices, accumulate, e, st);
        return launch_rd_fwd<ARITH, EPI_STORE, false>(p, image, out, nslices, accumulate, e, st);
    case EPI_RECIP:
        return launch_rd_fwd<ARITH, EPI_RECIP, true>(p, image, out, nslices, 0, e, st);
    case EPI_SIRT_FWD:
        return launch_rd_fwd<ARITH, EPI_SIRT_FWD, false>(p, image, out, nslices, 0, e, st);
    case EPI_MLEM_FWD:
        return launch_rd_fwd<ARITH, EPI_MLEM_FWD, false>(p, image, out, nslices, 0, e, st);
    case EPI_SPS_FWD:
        return launch_rd_fwd<ARITH, EPI_SPS_FWD, false>(p, image, out, nslices, 0, e, st);
    }
    return set_error(ITOMO_EINVAL, "rd forward: unsupported epilogue %d", epi);
}

}  // namespace

int rd_forward_epi(const Plan& p, int epi, int ones, const float* image, float* out,
                   int nslices, int accumulate, const EpiArgs& e, hipStream_t st,
                   int* blocks_per_slice)
{
    const int bps = ((p.npix + 63) / 64) * p.nang;
    if (blocks_per_slice) *blocks_per_slice = bps;
    EpiArgs ee = e;
    ee.blocks_per_slice = bps;
    int rc = p.arith == ITOMO_ARITH_FAST
                 ? dispatch_rd_fwd<ITOMO_ARITH_FAST>(p, epi, ones, image, out, nslices, accumulate, ee, st)
                 : dispatch_rd_fwd<ITOMO_ARITH_IEEE>(p, epi, ones, image, out, nslices, accumulate, ee, st);
    if (rc) return rc;
    return check_hip(hipGetLastError(), "rd forward launch");
}

// Back projection into `image` (overwritten, or accumulated into).
static int rd_back_launch(const Plan& p, int ones, const float* sino, float* image, int nslices,
                          int64_t sino_stride, int64_t img_stride, int accumulate,
                          hipStream_t st)
{
    if (p.rd_mat_state == 1) {
        rd_matrix_note_use(p, st);
        const int64_t n2 = (int64_t)p.npix * p.npix;
        dim3 mg((unsigned)((n2 + 63) / 64), nslices);
#define ITOMO_RDM(A, O)                                                                      \
    rd_back_matrix_kernel<A, O><<<mg, 64, 0, st>>>(p.rdb_ent, p.rdb_off, p.npix, sino, image, \
                                                   sino_stride, img_stride, accumulate)
        if (p.arith == ITOMO_ARITH_FAST) {
            if (ones) ITOMO_RDM(ITOMO_ARITH_FAST, true); else ITOMO_RDM(ITOMO_ARITH_FAST, false);
        } else {
            if (ones) ITOMO_RDM(ITOMO_ARITH_IEEE, true); else ITOMO_RDM(ITOMO_ARITH_IEEE, false);
        }
#undef ITOMO_RDM
        return check_hip(hipGetLastError(), "rd back (matrix) launch");
    }
    dim3 block(256), grid((p.npix + 15) / 16, (p.npix + 15) / 16, nslices);
    const RdView* g = (const RdView*)p.d_geom;
    if (p.arith == ITOMO_ARITH_FAST) {
        if (ones)
            rd_back_gather_kernel<ITOMO_ARITH_FAST, true><<<grid, block, 0, st>>>(
                g, p.nang, p.npix, sino, image, sino_stride, img_stride, accumulate);
        else
            rd_back_gather_kernel<ITOMO_ARITH_FAST, false><<<grid, block, 0, st>>>(
                g, p.nang, p.npix, sino, image, sino_stride, img_stride, accumulate);
    } else {
        if (ones)
            rd_back_gather_kernel<ITOMO_ARITH_IEEE, true><<<grid, block, 0, st>>>(
                g, p.nang, p.npix, sino, image, sino_stride, img_stride, accumulate);
        else
            rd_back_gather_kernel<ITOMO_ARITH_IEEE, false><<<grid, block, 0, st>>>(
                g, p.nang, p.npix, sino, image, sino_stride, img_stride, accumulate);
    }
    return check_hip(hipGetLastError(), "rd back launch");
}

int rd_back_overwrite(const Plan& p, int ones, const float* sino, float* image, int nslices,
                    hipStream_t st)
{
    return rd_back_launch(p, ones, sino, image, nslices, (int64_t)p.nang * p.npix,
                          (int64_t)p.npix * p.npix, 0, st);
}

int rd_forward(const Plan& p, const float* image, float* sino, int nslices, int64_t,
               int64_t, int accumulate, hipStream_t st)
{
    EpiArgs e{};
    return rd_forward_epi(p, EPI_STORE, 0, image, sino, nslices, accumulate, e, st, nullptr);
}

int rd_back(const Plan& p, const float* sino, float* image, int nslices, int64_t sino_stride,
            int64_t img_stride, int accumulate, hipStream_t st)
{
    return rd_back_launch(p, 0, sino, image, nslices, sino_stride, img_stride, accumulate, st);
}

}  // namespace itomo

extern "C" int itomo_plan_rd_matrix(itomo_plan* plan, int mode, size_t* bytes, void* stream)
{
    if (!plan || plan->projector != ITOMO_PROJ_RD || mode < ITOMO_RDM_QUERY ||
        mode > ITOMO_RDM_DROP)
        return itomo::set_error(ITOMO_EINVAL, "plan_rd_matrix: bad argument");
    int rc = ITOMO_OK;
    if (mode == ITOMO_RDM_BUILD) {
        if (itomo::scratch_region_active())
            return itomo::set_error(ITOMO_EINVAL, "plan_rd_matrix: inside a no-allocation call");
        if (plan->rd_mat_state == -1) plan->rd_mat_state = 0;
        rc = itomo::rd_matrix_ensure(*plan, (hipStream_t)stream);
    } else if (mode == ITOMO_RDM_DROP) {
        if (plan->rd_mat_pinned)
            return itomo::set_error(ITOMO_EINVAL, "plan_rd_matrix: a captured graph uses the "
                                                  "matrix; it stays until the plan is destroyed");
        rc = itomo::check_hip(hipStreamSynchronize((hipStream_t)stream), "plan_rd_matrix: sync");
        itomo::rd_matrix_free(*plan);
        plan->rd_mat_state = -1;
    }
    if (bytes) *bytes = plan->rd_mat_state == 1 ? plan->rd_mat_bytes : 0;
    return rc;
}
