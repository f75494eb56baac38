// Slant-stacking projector pair (semantics of radon_ss.c:43-196) for gfx950.
//
// Bin k = t + nh of view v is the line x c + y s = t; it goes to sinogram row nang-1-v.
// Views with |s| <= sqrt(1/2) step the image row u (y) and sample the column
// q = (t - u s)/c; the others step the column u (x) and sample the row q = (t - u c)/s.
// Each sample adds 1/|c| (or 1/|s|) times the image at the nearest pixel (method 0) or at
// floor(q) and floor(q)+1 with weights 1-w and w (method 1).  The stepped range of every
// bin (the reference's ray_limits and rounded loop bounds, radon_ss.c:43-88,121,159) is
// tabulated per plan on the host, clipped to the image: samples outside the square are
// skipped (the reference indexes outside the image rows there).
//
// Arithmetic is the reference's, operation for operation (ARITH FAST: its -ffast-math
// build; IEEE: the C as written); every update rounds to float after a double sum.
//   forward: one thread per bin steps u in order -- the reference's own loop;
//   back:    one thread per pixel gathers, per view in order, the up to 3 bins whose line
//            can reach it, in increasing t: each (view, bin) reaches a pixel at most once,
//            so the pixel receives the reference's terms in the reference's order.
// No atomics; both directions are bit-identical to the reference wherever its samples
// stay inside the image.
//
// Both wait for their gathers (a lane per bin reads the sampled index, so in the forward one of
// the two view families strides by rows): at 512^2 x 361 for 36% and 54% of the wave cycles, at
// 1.9 and 2.5 waves per SIMD, the VALU busy 42% and 28% of the time.  us before and after lockstep
// steps, the transposed copy and the two or three candidate bins, and now that the forward's
// steps without a pixel add -0 (see there), method 1: 64^2 x 45 views forward 19.1 -> 19.7 -> 11.6,
// back 43 -> 40; 257^2 x 180 91 -> 85 -> 43, 173 -> 148; 511^2 x 360 349 -> 235 -> 135, 397 -> 331;
// 512^2 x 361 x 2 slices 768 -> 309 -> 212, 540 -> 441; 1024^2 x 720 3176 -> 1125 -> 754, 2301 -> 1665.
#include "epilogue.h"

namespace itomo {

constexpr int kSsFwdBlock = 64;
constexpr int kSsBackX = 64, kSsBackY = 4;

// Sampled coordinate of stepped index u on line t (radon_ss.c:124,135,162,173).
template <int ARITH>
__device__ __forceinline__ float ss_q(const SsView& g, int u, float tf)
{
    if (ARITH == ITOMO_ARITH_FAST)  // (t - u a)/b as fma(-u, a, t) * (1/b)
        return __fmul_rn(__fmaf_rn(-(float)u, g.a, tf), g.rb);
    return __fsub_rn(__fdiv_rn(tf, g.b), __fdiv_rn(__fmul_rn((float)u, g.a), g.b));
}

template <int ARITH>
__device__ __forceinline__ int ss_round(float v)
{
    if (ARITH == ITOMO_ARITH_FAST)  // the fast build's float expansion of round()
        return (int)truncf(__fadd_rn(v, copysignf(0.49999997f, v)));
    return (int)round((double)v);
}

// Linear split of q: fl = floor(q), w = q - fl, wl = 1 - w as the build forms it.
template <int ARITH>
__device__ __forceinline__ void ss_split(float q, float& fl, float& w, float& wl)
{
    fl = floorf(q);
    w = __fsub_rn(q, fl);  // exact
    wl = (ARITH == ITOMO_ARITH_FAST) ? __fadd_rn(__fsub_rn(1.0f, q), fl) : __fsub_rn(1.0f, w);
}

// Forward update: bin + (w / |b|) * pix.
template <int ARITH>
__device__ __forceinline__ float ss_fwd_upd(float bin, float w, double rab, float pix)
{
    if (ARITH == ITOMO_ARITH_FAST)
        return (float)__fma_rn(__dmul_rn((double)w, rab), (double)pix, (double)bin);
    return (float)__dadd_rn((double)bin, __dmul_rn(__dmul_rn(rab, (double)w), (double)pix));
}

// Back update: pix + w * (bin / |b|).
template <int ARITH>
__device__ __forceinline__ float ss_back_upd(float pix, float w, double rab, float bin)
{
    if (ARITH == ITOMO_ARITH_FAST)
        return (float)__fma_rn((double)w, __dmul_rn((double)bin, rab), (double)pix);
    return (float)__dadd_rn((double)pix, __dmul_rn(__dmul_rn(rab, (double)w), (double)bin));
}

// Method-0 updates (weight 1): fma(v, 1/|b|, acc) in the fast build.
template <int ARITH>
__device__ __forceinline__ float ss_upd0(float acc, double rab, float v)
{
    if (ARITH == ITOMO_ARITH_FAST) return (float)__fma_rn((double)v, rab, (double)acc);
    return (float)__dadd_rn((double)acc, __dmul_rn(rab, (double)v));
}

// One thread per (sinogram row, bin).  Epilogues: STORE, RECIP.  The lanes of a wave, 64
// neighbouring bins, step the same u together, from the first lane's start to the last
// lane's end, and read the orientation in which the sampled index is contiguous (imageT, when
// there is one, for views that step columns): a wave's loads are then nearly contiguous, and
// four steps' loads are in flight before the first is added.  A bin's sum is one serial chain: a
// step outside the bin's range or the image adds -0, which leaves any sum as it is, where a
// select after every addition lengthened the chain (and small calls, 3-5% slower by it).
template <int ARITH, int METHOD, int EPI, bool ONES>
__global__ void __launch_bounds__(kSsFwdBlock)
ss_fwd_kernel(const SsView* __restrict__ geom, const int2* __restrict__ range, int npix,
              int nang, const float* __restrict__ image, const float* __restrict__ imageT,
              float* __restrict__ out, int64_t img_stride, int64_t sino_stride, int accumulate,
              EpiArgs e)
{
    constexpr int U = 4;
    const int k = blockIdx.x * kSsFwdBlock + threadIdx.x;
    const bool active = k < npix;
    const int r = blockIdx.y, z = blockIdx.z;
    const int v = nang - 1 - r;
    const int64_t soff = (int64_t)z * sino_stride, o = (int64_t)r * npix + k;
    float acc = (EPI == EPI_STORE && accumulate && active) ? out[soff + o] : 0.0f;
    const int nh = npix >> 1;
    const SsView g = geom[v];
    // odd npix: the last bin has no line (radon_ss.c:109)
    int2 ur = make_int2(0, 0);
    if (k < 2 * nh) ur = range[(int64_t)v * npix + k];
    int first = ur.x < ur.y ? ur.x : npix, last = ur.x < ur.y ? ur.y : -npix;
    for (int off = 32; off > 0; off >>= 1) {
        first = min(first, __shfl_xor(first, off, 64));
        last = max(last, __shfl_xor(last, off, 64));
    }
    const float tf = (float)(k - nh);
    // stepped index u -> image (stepped, sampled) strides
    const bool flip = imageT && !g.ybranch;
    const float* __restrict__ img = (flip ? imageT : image) + (int64_t)z * img_stride;
    const int ss = g.ybranch || flip ? npix : 1, sq = g.ybranch || flip ? 1 : npix;
    for (int u0 = first; u0 < last; u0 += U) {
        float fa[U], fb[U], wa[U], wb[U];
#pragma unroll
        for (int c = 0; c < U; ++c) {
            const int u = u0 + c;
            const bool in = u >= ur.x && u < ur.y;
            const float q = ss_q<ARITH>(g, u, tf);
            const float* __restrict__ line = img + (unsigned)((u + nh) * ss);
            // what is added where there is no pixel: any sum plus -0 is that sum
            fa[c] = fb[c] = -0.0f;
            wa[c] = wb[c] = 1.0f;
            if (METHOD == 0) {
                const int p = ss_round<ARITH>(q) + nh;
                if (in && p >= 0 && p < npix) fa[c] = ONES ? 1.0f : line[__umul24(p, sq)];
            } else {
                float fl, w, wl;
                ss_split<ARITH>(q, fl, w, wl);
                const int p = (int)fl + nh;
                if (in && p >= 0 && p <= npix - 1) fa[c] = ONES ? 1.0f : line[__umul24(p, sq)];
                if (in && p + 1 >= 0 && p + 1 <= npix - 1)
                    fb[c] = ONES ? 1.0f : line[__umul24(p + 1, sq)];
                wa[c] = wl;
                wb[c] = w;
            }
        }
#pragma unroll
        for (int c = 0; c < U; ++c) {
            if (METHOD == 0) {
                acc = ss_upd0<ARITH>(acc, g.rab, fa[c]);
            } else {
                acc = ss_fwd_upd<ARITH>(acc, wa[c], g.rab, fa[c]);
                acc = ss_fwd_upd<ARITH>(acc, wb[c], g.rab, fb[c]);
            }
        }
    }
    double p0 = 0.0;
    if (active) out[soff + o] = epi_forward<EPI>(acc, o, soff, z, e, &p0);
}

// One thread per pixel (memory row R, column Q); 64 columns x 4 rows per block.
template <int ARITH, int METHOD, int EPI, bool ONES>
__global__ void __launch_bounds__(kSsBackX * kSsBackY)
ss_back_kernel(const SsView* __restrict__ geom, const int2* __restrict__ range, int npix,
               int nang, const float* __restrict__ sino, float* __restrict__ out,
               int64_t sino_stride, int64_t img_stride, int accumulate, EpiArgs e)
{
    const int Q = blockIdx.x * kSsBackX + threadIdx.x;
    const int R = blockIdx.y * kSsBackY + threadIdx.y;
    const int z = blockIdx.z;
    sino += (int64_t)z * sino_stride;
    const int64_t ioff = (int64_t)z * img_stride, o = (int64_t)R * npix + Q;
    double p1 = 0.0, p2 = 0.0;
    if (Q < npix && R < npix) {
        const int nh = npix >> 1;
        // Bins whose line passes within |b| (and a margin) of the pixel centre in the sampled
        // coordinate, t = u a + q b with q in [P - 1, P + 1]: the integers within |b| <= 1 of
        // tc = u a + P b, so two of them, or three where |b| is within the margin of 1 (float
        // rounding of tc and q stays below npix * 2^-21).  Each is then decided exactly.  A
        // pixel two or more pixels inside the image needs no look at the bins' ranges: a line
        // that samples next to it enters and leaves the square at least one step from u.
        const float margin = 0.01f + npix * 0x1p-18f;
        float acc = (EPI == EPI_STORE && accumulate) ? out[ioff + o] : 0.0f;
        const bool inner = Q >= 2 && R >= 2 && Q < 2 * nh - 3 && R < 2 * nh - 3;
        for (int v = 0; v < nang; ++v) {
            const SsView g = geom[v];
            const int u = (g.ybranch ? R : Q) - nh;  // stepped
            const int P = (g.ybranch ? Q : R) - nh;  // sampled
            const float tc = __builtin_fmaf((float)u, g.a, __fmul_rn((float)P, g.b));
            const float hw = __builtin_fmaf(fabsf(g.b), 1.0f + margin, margin);
            const float tf = ceilf(tc - hw);
            const float* __restrict__ row = sino + (int64_t)(nang - 1 - v) * npix;
            const int2* __restrict__ rg = range + (int64_t)v * npix;
            float wt[3], val[3];
            bool ok[3];
            auto look = [&](int c) {
                const float tcf = __fadd_rn(tf, (float)c);
                const int t = (int)tcf, k = t + nh;
                ok[c] = t >= -nh && t < nh;
                const float q = ss_q<ARITH>(g, u, tcf);
                if (METHOD == 0) {
                    ok[c] = ok[c] && ss_round<ARITH>(q) == P;
                    wt[c] = 1.0f;
                } else {
                    float fl, w, wl;
                    ss_split<ARITH>(q, fl, w, wl);
                    const int p = (int)fl;
                    ok[c] = ok[c] && (p == P || p + 1 == P);
                    wt[c] = p == P ? wl : w;
                }
                if (!inner && ok[c]) {
                    const int2 ur = rg[k];
                    ok[c] = u >= ur.x && u < ur.y;
                }
                val[c] = ONES || !ok[c] ? 1.0f : row[k];
            };
            auto add = [&](int c) {
                const float na = METHOD == 0 ? ss_upd0<ARITH>(acc, g.rab, val[c])
                                             : ss_back_upd<ARITH>(acc, wt[c], g.rab, val[c]);
                acc = ok[c] ? na : acc;
            };
            look(0);
            look(1);
            const bool third = __any(tf + 2.0f <= tc + hw);
            if (third) look(2);
            add(0);
            add(1);
            if (third) add(2);
        }
        const float xo = epi_updates_x(EPI) ? out[ioff + o] : 0.0f;
        out[ioff + o] = epi_back<EPI>(acc, xo, o, z, e, &p1, &p2);
    }
    if (epi_has_partials(EPI) && e.partials) {
        const int blk = blockIdx.y * gridDim.x + blockIdx.x;
        block_partials3(0.0, p1, p2, e.partials + ((int64_t)z * e.blocks_per_slice + blk) * 3);
    }
}

namespace {

template <int ARITH, int METHOD, int EPI, bool ONES>
void launch_ss_fwd(const Plan& p, const float* image, const float* imageT, float* out,
                   int nslices, int accumulate, const EpiArgs& e, hipStream_t st)
{
    dim3 grid((p.npix + kSsFwdBlock - 1) / kSsFwdBlock, p.nang, nslices);
    ss_fwd_kernel<ARITH, METHOD, EPI, ONES><<<grid, kSsFwdBlock, 0, st>>>(
        (const SsView*)p.d_geom, (const int2*)p.d_range, p.npix, p.nang, image, imageT, out,
        (int64_t)p.npix * p.npix, (int64_t)p.nang * p.npix, accumulate, e);
}

template <int ARITH, int METHOD>
int dispatch_ss_fwd(const Plan& p, int epi, int ones, const float* image, const float* imageT,
                    float* out, int nslices, int accumulate, const EpiArgs& e, hipStream_t st)
{
    if (epi == EPI_STORE) {
        if (ones) launch_ss_fwd<ARITH, METHOD, EPI_STORE, true>(p, image, imageT, out, nslices, accumulate, e, st);
        else launch_ss_fwd<ARITH, METHOD, EPI_STORE, false>(p, image, imageT, out, nslices, accumulate, e, st);
        return ITOMO_OK;
    }
    if (epi == EPI_RECIP && ones) {
        launch_ss_fwd<ARITH, METHOD, EPI_RECIP, true>(p, image, imageT, out, nslices, 0, e, st);
        return ITOMO_OK;
    }
    return set_error(ITOMO_EINVAL, "ss forward: unsupported epilogue %d", epi);
}

template <int ARITH, int METHOD, int EPI, bool ONES>
void launch_ss_back(const Plan& p, const float* sino, float* out, int nslices, int accumulate,
                    const EpiArgs& e, hipStream_t st)
{
    dim3 block(kSsBackX, kSsBackY);
    dim3 grid((p.npix + kSsBackX - 1) / kSsBackX, (p.npix + kSsBackY - 1) / kSsBackY, nslices);
    ss_back_kernel<ARITH, METHOD, EPI, ONES><<<grid, block, 0, st>>>(
        (const SsView*)p.d_geom, (const int2*)p.d_range, p.npix, p.nang, sino, out,
        (int64_t)p.nang * p.npix, (int64_t)p.npix * p.npix, accumulate, e);
}

template <int ARITH, int METHOD>
int dispatch_ss_back(const Plan& p, int epi, int ones, const float* sino, float* out,
                     int nslices, int accumulate, const EpiArgs& e, hipStream_t st)
{
    switch (epi) {
    case EPI_STORE:
        if (ones) launch_ss_back<ARITH, METHOD, EPI_STORE, true>(p, sino, out, nslices, accumulate, e, st);
        else launch_ss_back<ARITH, METHOD, EPI_STORE, false>(p, sino, out, nslices, accumulate, e, st);
        return ITOMO_OK;
    case EPI_RECIP:
        if (!ones) break;
        launch_ss_back<ARITH, METHOD, EPI_RECIP, true>(p, sino, out, nslices, 0, e, st);
        return ITOMO_OK;
    case EPI_SIRT_BACK:
        launch_ss_back<ARITH, METHOD, EPI_SIRT_BACK, false>(p, sino, out, nslices, 0, e, st);
        return ITOMO_OK;
    case EPI_MLEM_BACK:
        launch_ss_back<ARITH, METHOD, EPI_MLEM_BACK, false>(p, sino, out, nslices, 0, e, st);
        return ITOMO_OK;
    case EPI_SPS_BACK:
        launch_ss_back<ARITH, METHOD, EPI_SPS_BACK, false>(p, sino, out, nslices, 0, e, st);
        return ITOMO_OK;
    }
    return set_error(ITOMO_EINVAL, "ss back: unsupported epilogue %d", epi);
}

}  // namespace

int ss_forward_epi(const Plan& p, int epi, int ones, const float* image, float* out,
                   int nslices, int accumulate, const EpiArgs& e, hipStream_t st,
                   int* blocks_per_slice)
{
    if (epi == EPI_SIRT_FWD || epi == EPI_SPS_FWD || epi == EPI_MLEM_FWD) {
        int rc = ss_forward_epi(p, EPI_STORE, ones, image, out, nslices, 0, EpiArgs{}, st,
                                nullptr);
        if (rc) return rc;
        return elementwise_fwd_epilogue(epi, out, e, (int64_t)p.nang * p.npix, nslices, st,
                                        blocks_per_slice);
    }
    if (blocks_per_slice) *blocks_per_slice = 0;
    for (int z = 0; z < nslices;) {
        const float* im = image ? image + (int64_t)z * p.npix * p.npix : nullptr;
        float* o = out + (int64_t)z * p.nang * p.npix;
        const TransposedCopy tc(p, !ones, im, nslices - z, st);
        const float* imT = tc.get();
        const int n = tc.slices();
        int rc;
        if (p.arith == ITOMO_ARITH_FAST)
            rc = p.method == 0
                     ? dispatch_ss_fwd<ITOMO_ARITH_FAST, 0>(p, epi, ones, im, imT, o, n, accumulate, e, st)
                     : dispatch_ss_fwd<ITOMO_ARITH_FAST, 1>(p, epi, ones, im, imT, o, n, accumulate, e, st);
        else
            rc = p.method == 0
                     ? dispatch_ss_fwd<ITOMO_ARITH_IEEE, 0>(p, epi, ones, im, imT, o, n, accumulate, e, st)
                     : dispatch_ss_fwd<ITOMO_ARITH_IEEE, 1>(p, epi, ones, im, imT, o, n, accumulate, e, st);
        if (rc) return rc;
        z += n;
    }
    return check_hip(hipGetLastError(), "ss forward launch");
}

int ss_back_epi(const Plan& p, int epi, int ones, const float* sino, float* out, int nslices,
                int accumulate, const EpiArgs& e, hipStream_t st, int* blocks_per_slice)
{
    const int bps = (int)back_blocks_per_slice(p, nslices);
    if (blocks_per_slice) *blocks_per_slice = bps;
    EpiArgs ee = e;
    ee.blocks_per_slice = bps;
    int rc;
    if (p.arith == ITOMO_ARITH_FAST)
        rc = p.method == 0
                 ? dispatch_ss_back<ITOMO_ARITH_FAST, 0>(p, epi, ones, sino, out, nslices, accumulate, ee, st)
                 : dispatch_ss_back<ITOMO_ARITH_FAST, 1>(p, epi, ones, sino, out, nslices, accumulate, ee, st);
    else
        rc = p.method == 0
                 ? dispatch_ss_back<ITOMO_ARITH_IEEE, 0>(p, epi, ones, sino, out, nslices, accumulate, ee, st)
                 : dispatch_ss_back<ITOMO_ARITH_IEEE, 1>(p, epi, ones, sino, out, nslices, accumulate, ee, st);
    if (rc) return rc;
    return check_hip(hipGetLastError(), "ss back launch");
}

int ss_forward(const Plan& p, const float* image, float* sino, int nslices, int64_t, int64_t,
               int accumulate, hipStream_t st)
{
    return ss_forward_epi(p, EPI_STORE, 0, image, sino, nslices, accumulate, EpiArgs{}, st,
                          nullptr);
}

int ss_back(const Plan& p, const float* sino, float* image, int nslices, int64_t, int64_t,
            int accumulate, hipStream_t st)
{
    return ss_back_epi(p, EPI_STORE, 0, sino, image, nslices, accumulate, EpiArgs{}, st,
                       nullptr);
}

}  // namespace itomo
