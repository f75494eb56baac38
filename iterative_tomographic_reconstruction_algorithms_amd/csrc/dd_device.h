// Device code of the distance-driven projector pair, shared by the per-plan kernels
// (dd.hip) and the persistent batch kernels (batch.hip).
#pragma once

#include "epilogue.h"

namespace itomo {

namespace {

// Bin boundary D for j = d - nh, with j given as an integer-valued float.
template <int ARITH>
__device__ __forceinline__ float key_Df(const DdView& g, float x)
{
    if (ARITH == ITOMO_ARITH_FAST) return __fmul_rn(x, g.rinv);
    return __fdiv_rn(x, g.b);
}

template <int ARITH>
__device__ __forceinline__ float key_D(const DdView& g, int j)
{
    return key_Df<ARITH>(g, (float)j);
}

// Line offset K for line coordinate u = (i - nh) + 0.5.
template <int ARITH>
__device__ __forceinline__ float key_K(const DdView& g, float u)
{
    if (ARITH == ITOMO_ARITH_FAST) return __fmul_rn(u, g.t);
    return __fdiv_rn(__fmul_rn(u, g.a), g.b);
}

__device__ __forceinline__ float line_coord(int i, int nh) { return (float)(i - nh) + 0.5f; }

// acc += w * v as the reference build evaluates it: fused under -ffast-math (FAST),
// a rounded product then a rounded sum as written (IEEE).
template <int ARITH>
__device__ __forceinline__ float accum(float w, float v, float acc)
{
    if (ARITH == ITOMO_ARITH_FAST) return __builtin_fmaf(w, v, acc);
    return __fadd_rn(acc, __fmul_rn(w, v));
}

// Start L* of the segment a sweep line drops (radon_dd.c:176-177).  The reference
// merges the pixel keys P_0..P_N with the bin keys D_0..D_N (on equal keys the pixel
// key first) and stops at the first key with index N, before that segment is used;
// L* is the key merged just before it:
//   P_N <= D_N (stop at P_N):  L* = max(P_{N-1}, largest D_j <  P_N)
//   D_N <  P_N (stop at D_N):  L* = max(D_{N-1}, largest P_k <= D_N)
// Every other segment ends at or before L*, so clipping each segment's right end to L*
// removes exactly the dropped one -- also when P_k == D_N for some k < N, where the
// dropped segment has zero length and the one ending at P_k is kept.
template <int ARITH>
__device__ __forceinline__ float dd_line_end(const DdView& g, int npix, int nh, int i)
{
    const float K = key_K<ARITH>(g, line_coord(i, nh));
    const float PN = __fsub_rn((float)(npix - nh), K);
    const float DN = key_D<ARITH>(g, npix - nh);
    const float ninf = __int_as_float(0xff800000);
    // binary search for the last index in [0, npix) whose key precedes the stop key;
    // both key sequences are non-decreasing in their index
    int lo = -1, hi = npix;
    if (PN <= DN) {
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (key_D<ARITH>(g, mid - nh) < PN) lo = mid; else hi = mid;
        }
        const float Dj = lo >= 0 ? key_D<ARITH>(g, lo - nh) : ninf;
        return fmaxf(__fsub_rn((float)(npix - 1 - nh), K), Dj);
    }
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (__fsub_rn((float)(mid - nh), K) <= DN) lo = mid; else hi = mid;
    }
    const float Pk = lo >= 0 ? __fsub_rn((float)(lo - nh), K) : ninf;
    return fmaxf(key_D<ARITH>(g, npix - 1 - nh), Pk);
}

}  // namespace

// ---- back projection ----------------------------------------------------------------
//
// Block = T x T pixel tile, (T/P)^2 threads, each thread a P x P micro-tile (rows
// P*ty.., columns P*tx..).  For a row sweep a thread walks its P rows, P consecutive
// pixels each; for a column sweep its P columns.  Along one line the bin walk is
// incremental: the first pixel's bin is found once, then each next pixel continues from
// the previous pixel's last bin.  Views are processed in chunks of back_views: the
// sinogram values the tile can touch in each view (at most back_foot(T) bins) are staged
// in LDS, with zeros for bins outside [0, npix), so the walk needs no bounds checks.  The
// accumulation order per pixel (views in list order, bins increasing) is the reference's
// for every (T, P), so all tilings give bit-identical images.
template <int T, int P>
constexpr int back_views()
{
    return T / P == 8 ? 512 / T : (T == 16 ? 64 : 32);
}

// Staged bins per view: the tile's footprint spans T*(|sin|+|cos|) <= T*sqrt(2) bins,
// plus 7 for the floors and the +-2 margins of staged_range.
template <int T>
constexpr int back_foot() { return (T * 1449) / 1024 + 10; }

// What a tile needs of a view: nothing (it projects outside the detector, or no branch of
// the reference takes the view), the walk without or with the clip to L*, the walk for views
// where a pixel may hold two bin keys (with the clip), or a plain sum.
enum BackClass : int { BACK_SKIP = 0, BACK_WALK, BACK_CLIP, BACK_MULTI, BACK_SUM };

// The class of view g for a tile, and the bins it can touch: the first one, *b_lo, which may
// lie outside the detector (staged as zeros, so the walks need no clamp), and their number.
// L* >= min(P[N-1], D[N-1]) on every line, so it clips nothing where the tile's pixels all
// lie before the last pixel of their lines and project inside the bins [0, npix - 1).
template <int ARITH, int T>
__device__ __forceinline__ int staged_range(const DdView& g, int npix, int nh, int r0, int q0,
                                            int* b_lo, int* cnt)
{
    *b_lo = 0;
    *cnt = 0;
    if (g.kind == DD_ROWSUM || g.kind == DD_COLSUM) {
        *b_lo = g.kind == DD_ROWSUM ? r0 : q0;
        *cnt = T;
        return BACK_SUM;
    }
    if (g.kind != DD_SWEEP_ROWS && g.kind != DD_SWEEP_COLS) return BACK_SKIP;
    // lines are rows (r) or columns (q); pixel boundaries along the line
    const int l0 = (g.kind == DD_SWEEP_ROWS) ? r0 : q0;
    const int p0 = (g.kind == DD_SWEEP_ROWS) ? q0 : r0;
    const float ka = (float)(l0 - nh) + 0.5f, kb = ka + (float)(T - 1);
    const float K1 = ka * g.t, K2 = kb * g.t;
    const float kmin = (float)(p0 - nh) - fmaxf(K1, K2);
    const float kmax = (float)(p0 + T - nh) - fminf(K1, K2);
    const int lo = (int)floorf(kmin * g.est) + nh - 2;
    const int hi = (int)floorf(kmax * g.est) + nh + 2;
    if (hi < 0 || lo >= npix) return BACK_SKIP;
    *b_lo = lo;
    *cnt = min(hi - lo + 1, back_foot<T>());
    if (g.multi) return BACK_MULTI;
    return hi <= npix - 2 && p0 + T < npix ? BACK_WALK : BACK_CLIP;
}

// Constants of a walked view as the walk reads them from LDS: (rinv, t) in FAST
// and (b, a) in IEEE arithmetic, est, and the index offset of the view's staged bins.
template <int ARITH>
__device__ __forceinline__ float4 walk_pack(const DdView& g, int base)
{
    if (ARITH == ITOMO_ARITH_FAST) return make_float4(g.rinv, g.t, g.est, __int_as_float(base));
    return make_float4(g.b, g.a, g.est, __int_as_float(base));
}

template <int ARITH>
__device__ __forceinline__ DdView walk_unpack(float4 c)
{
    DdView g;
    if (ARITH == ITOMO_ARITH_FAST) {
        g.rinv = c.x;
        g.t = c.y;
    } else {
        g.b = c.x;
        g.a = c.y;
    }
    g.est = c.z;
    return g;
}

// jr = (index - nh) of the right key of the bin that holds a pixel's left end lo
// (D_jr-1 <= lo < D_jr).  In index units the estimate lo*est is off from lo/(bin width) by a
// relative 2^-22 (est * rinv = 1 + 2^-23 at most) and the keys by a relative 2^-24; with
// |j| <= 2*16384 that stays below 0.01, so floor(lo*est + 1/2) is the bin or the one after it
// and one test against its key settles it.
template <int ARITH>
__device__ __forceinline__ int walk_first(const DdView& g, float lo)
{
    float fd = floorf(__fadd_rn(__fmul_rn(lo, g.est), 0.5f));
    // the integer comes from this very float: left to itself the compiler fuses the rounded
    // sum, the floor and the conversion into an instruction that rounds otherwise
    asm("" : "+v"(fd));
    int jr = (int)fd + 1;
    jr -= lo < key_Df<ARITH>(g, fd);
    return jr;
}

// The P x P pixels of a thread in a walked view (see staged_range): lines u, u + 1, ... and
// along each line the pixels from x0; pixel k of line i goes to a[i * LS + k * KS].  S[jr] is
// the value of the bin whose right key has index jr (zero outside the detector); Ls[i] is
// L* of line i.  A pixel [lo, hi] gives that bin the weight m - lo and the next one hi - m with
// m = min(hi, Dhi): where it does not reach past Dhi the second is exactly 0, where it does
// they are that pixel's own overlaps, end minus start.  (Bins are at least as wide as pixels,
// so a pixel reaches one bin key at most, except where the two widths agree to rounding:
// MULTI takes a third bin the same way; three keys in a pixel would need bins of half a
// pixel.)  CLIP: hi is clipped to L* first, and a pixel that starts past L* gets the weight 0.
// A weight of 0 leaves the sum unchanged, so no overlap needs a test.  11 VALU operations per
// pixel, CLIP 13.  The lines advance side by side, and a step's values are added one step
// later, so that the P chains (key, compare, next bin) and the LDS reads hide behind each
// other.
template <int ARITH, int P, int LS, int KS, bool CLIP, bool MULTI = false>
__device__ __forceinline__ void walk_tile(const DdView& g, float u, float x0, const float* S,
                                          const float* Ls, float* a)
{
    // taken anew per call: the compiler would otherwise keep every u + i and x0 + k of both
    // sweep directions in registers across the views
    asm("" : "+v"(u), "+v"(x0));
    float K[P], lo[P], end[P];
    int jr[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        K[i] = key_K<ARITH>(g, __fadd_rn(u, (float)i));
        lo[i] = __fsub_rn(x0, K[i]);
        jr[i] = walk_first<ARITH>(g, lo[i]);
        if (CLIP) end[i] = Ls[i];
    }
    float w0[P], w1[P], w2[P], s0[P], s1[P], s2[P];
#pragma unroll
    for (int k = 0; k <= P; ++k) {
        float v0[P], v1[P], v2[P], t0[P], t1[P], t2[P];
        if (k < P) {
#pragma unroll
            for (int i = 0; i < P; ++i) {
                t0[i] = S[jr[i]];
                t1[i] = S[jr[i] + 1];
                const float Dhi = key_Df<ARITH>(g, (float)jr[i]);
                const float hi = __fsub_rn(__fadd_rn(x0, (float)(k + 1)), K[i]);
                const float hc = CLIP ? fminf(hi, end[i]) : hi;
                const float m = fminf(hc, Dhi);
                v0[i] = __fsub_rn(m, lo[i]);
                if (CLIP) v0[i] = fmaxf(v0[i], 0.0f);
                if (MULTI) {
                    const float Dhi2 = key_Df<ARITH>(g, (float)(jr[i] + 1));
                    const float m2 = fminf(hc, Dhi2);
                    const float third = S[jr[i] + 2];   // read by every lane, used by few
                    v1[i] = fmaxf(__fsub_rn(m2, Dhi), 0.0f);
                    v2[i] = __fsub_rn(hc, m2);
                    t2[i] = Dhi2 < hc ? third : 0.0f;
                    jr[i] += Dhi2 < hi;
                } else {
                    v1[i] = __fsub_rn(hc, m);
                }
                jr[i] += Dhi < hi;
                // kept as one value (a carry add): the compiler would otherwise track the
                // LDS address and the key's index apart
                asm("" : "+v"(jr[i]));
                lo[i] = hi;
            }
        }
        if (k > 0) {
#pragma unroll
            for (int i = 0; i < P; ++i) {
                float& acc = a[i * LS + (k - 1) * KS];
                acc = accum<ARITH>(w0[i], s0[i], acc);
                acc = accum<ARITH>(w1[i], s1[i], acc);
                if (MULTI) acc = accum<ARITH>(w2[i], s2[i], acc);
            }
        }
#pragma unroll
        for (int i = 0; i < P; ++i) {
            w0[i] = v0[i];
            w1[i] = v1[i];
            s0[i] = t0[i];
            s1[i] = t1[i];
            if (MULTI) {
                w2[i] = v2[i];
                s2[i] = t2[i];
            }
        }
    }
}

// A wave-uniform 64-bit value as scalars.
__device__ __forceinline__ unsigned long long uniform64(unsigned long long m)
{
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)m);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(unsigned)(m >> 32));
    return lo | (unsigned long long)hi << 32;
}

// One T x T tile (tile column bx, tile row by) of slice z; blk indexes its FP64
// partials.  Shared by the per-plan kernel and the persistent batch kernel.
template <int ARITH, int EPI, bool ONES, int T, int P>
__device__ __forceinline__ void dd_back_tile(const DdView* __restrict__ geom,
                                             const float* __restrict__ lstar, int nang, int npix,
                                             const float* __restrict__ sino,
                                             float* __restrict__ out, int64_t sino_stride,
                                             int64_t img_stride, int accumulate,
                                             const EpiArgs& e, int bx, int by, int z, int blk)
{
    constexpr int TP = T / P, NT = TP * TP, FOOT = back_foot<T>(), kBackViews = back_views<T, P>();
    __shared__ float sS[kBackViews][FOOT];
    __shared__ int sLo[kBackViews];
    __shared__ int sCnt[kBackViews];
    __shared__ int sRow[kBackViews];
    __shared__ int sLine[kBackViews];
    __shared__ float4 sGeo[kBackViews];      // walked views: see walk_pack
    // bit v: view v of the chunk is walked, walked with the clip, skipped, sweeps rows, has
    // two keys in a pixel
    __shared__ unsigned long long sMask[5];
    __shared__ float sLs[kBackViews][T];   // L* of the tile's lines per view

    const int tid = threadIdx.x;
    // Threads -> micro-tiles: each wave takes an 8 x 8 block of micro-tiles (2 x 2 waves
    // per 16 x 16 block), so the 32 lanes of a half-wave cover a 32 x 16-pixel patch
    // (P = 4) whose projection onto the detector spans at most 28|c| + 12|s| < 31 bins:
    // the staged bins they read in one step lie in distinct LDS banks.  (Rows of 16
    // micro-tiles per half-wave span up to 60 bins and conflicted.)
    static_assert(TP == 8 || TP == 16, "micro-tile grid");
    const int lane = tid & 63, wv = tid >> 6;
    const int tx = TP == 16 ? ((wv & 1) << 3) + (lane & 7) : tid % TP;
    const int ty = TP == 16 ? ((wv >> 1) << 3) + (lane >> 3) : tid / TP;
    const int r0 = by * T, q0 = bx * T;
    const int rr = r0 + P * ty, cc = q0 + P * tx;  // micro-tile origin
    sino += (int64_t)z * sino_stride;
    out += (int64_t)z * img_stride;
    const int nh = (int)(npix * 0.5);

    float acc[P][P];
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int r = rr + i, q = cc + j;
            acc[i][j] = (EPI == EPI_STORE && accumulate && r < npix && q < npix)
                            ? out[(int64_t)r * npix + q]
                            : 0.0f;
        }
    // With small micro-tiles the epilogue inputs (current iterate and weight) are
    // loaded up front, so their latency hides behind the view loop.
    constexpr bool PRE = P <= 2 && (epi_updates_x(EPI) || epi_back_uses_w(EPI));
    float pre_x[P][P], pre_w[P][P];
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
        for (int j = 0; j < P; ++j) {
            pre_x[i][j] = 0.0f;
            pre_w[i][j] = 0.0f;
            const int r = rr + i, q = cc + j;
            if (PRE && r < npix && q < npix) {
                const int64_t o = (int64_t)r * npix + q;
                if (epi_updates_x(EPI)) pre_x[i][j] = out[o];
                if (epi_back_uses_w(EPI)) pre_w[i][j] = e.w[(int64_t)z * e.w_stride + o];
            }
        }

    for (int v0 = 0; v0 < nang; v0 += kBackViews) {
        const int nv = min(kBackViews, nang - v0);
        __syncthreads();  // previous chunk fully consumed
        if (tid < 64) {
            int cls = BACK_SKIP;
            bool rows = false;
            if (tid < nv) {
                int lo, cnt;
                const DdView g = geom[v0 + tid];
                cls = staged_range<ARITH, T>(g, npix, nh, r0, q0, &lo, &cnt);
                sLo[tid] = lo;
                sCnt[tid] = cnt;
                sRow[tid] = g.row;
                sLine[tid] = g.kind == DD_SWEEP_COLS ? q0 : r0;
                rows = g.kind == DD_SWEEP_ROWS;
                sGeo[tid] = walk_pack<ARITH>(g, tid * FOOT - lo + nh - 1);
            }
            const unsigned long long b0 = __ballot(cls == BACK_WALK || cls == BACK_CLIP),
                                     b1 = __ballot(cls == BACK_CLIP),
                                     b2 = __ballot(cls == BACK_SKIP), b3 = __ballot(rows),
                                     b4 = __ballot(cls == BACK_MULTI);
            if (tid == 0) {
                sMask[0] = b0;
                sMask[1] = b1;
                sMask[2] = b2;
                sMask[3] = b3;
                sMask[4] = b4;
            }
        }
        __syncthreads();
        const unsigned long long walked = uniform64(sMask[0]), clipped = uniform64(sMask[1]),
                                 skipped = uniform64(sMask[2]), rowviews = uniform64(sMask[3]),
                                 multi = uniform64(sMask[4]);
        // Four loads at a time: one by one, each waits for its own latency at the barriers'
        // expense; all at once, they take the registers of the walk.
        constexpr int U = NT == 64 ? 8 : 4;
#pragma unroll 1
        for (int k0 = tid; k0 < nv * FOOT; k0 += U * NT) {
            float val[U];
#pragma unroll
            for (int r = 0; r < U; ++r) {
                const int k = k0 + r * NT, v = k / FOOT, j = k - v * FOOT;
                val[r] = 0.0f;
                if (v < nv) {
                    const int d = sLo[v] + j;
                    if (j < sCnt[v] && d >= 0 && d < npix)
                        val[r] = ONES ? 1.0f : sino[(int64_t)sRow[v] * npix + d];
                }
            }
#pragma unroll
            for (int r = 0; r < U; ++r)
                if (k0 + r * NT < nv * FOOT) (&sS[0][0])[k0 + r * NT] = val[r];
        }
#pragma unroll 1
        for (int k0 = tid; k0 < nv * T; k0 += U * NT) {
            float val[U];
#pragma unroll
            for (int r = 0; r < U; ++r) {
                const int k = k0 + r * NT, v = k / T, l = k - v * T;
                val[r] = INFINITY;   // no clip
                if (v < nv && !(((walked & ~clipped) | skipped) >> v & 1)) {
                    const int line = sLine[v] + l;
                    if (line < npix) val[r] = lstar[(int64_t)(v0 + v) * npix + line];
                }
            }
#pragma unroll
            for (int r = 0; r < U; ++r)
                if (k0 + r * NT < nv * T) (&sLs[0][0])[k0 + r * NT] = val[r];
        }
        __syncthreads();
        for (int v = 0; v < nv; ++v) {
            if ((skipped >> v) & 1) continue;
            if constexpr (P == 1) {
                // One pixel per thread: G consecutive walked views are formed side by side and
                // added in view order.
                constexpr int G = 4;
                constexpr unsigned ALL = (1u << G) - 1;
                if (v + G <= nv && ((walked >> v) & ALL) == ALL) {
                    float wa[G], wb[G], sa[G], sb[G];
                    const bool clip = ((clipped >> v) & ALL) != 0;
#pragma unroll
                    for (int k = 0; k < G; ++k) {
                        const float4 c = sGeo[v + k];
                        const DdView g = walk_unpack<ARITH>(c);
                        const float* S = &sS[0][0] + __float_as_int(c.w);
                        const bool rows = (rowviews >> (v + k)) & 1;
                        const float K = key_K<ARITH>(g, line_coord(rows ? rr : cc, nh));
                        const float x = (float)((rows ? cc : rr) - nh);
                        const float lo = __fsub_rn(x, K);
                        const int jr = walk_first<ARITH>(g, lo);
                        sa[k] = S[jr];
                        sb[k] = S[jr + 1];
                        float hi = __fsub_rn(__fadd_rn(x, 1.0f), K);
                        if (clip) hi = fminf(hi, sLs[v + k][rows ? ty : tx]);
                        const float m = fminf(hi, key_Df<ARITH>(g, (float)jr));
                        wa[k] = fmaxf(__fsub_rn(m, lo), 0.0f);
                        wb[k] = __fsub_rn(hi, m);
                    }
#pragma unroll
                    for (int k = 0; k < G; ++k) {
                        acc[0][0] = accum<ARITH>(wa[k], sa[k], acc[0][0]);
                        acc[0][0] = accum<ARITH>(wb[k], sb[k], acc[0][0]);
                    }
                    v += G - 1;
                    continue;
                }
            }
            if (((walked | multi) >> v) & 1) {
                const float4 c = sGeo[v];
                const DdView g = walk_unpack<ARITH>(c);
                const float* S = &sS[0][0] + __float_as_int(c.w);
                if ((rowviews >> v) & 1) {
                    const float u = line_coord(rr, nh), x0 = (float)(cc - nh);
                    const float* Ls = &sLs[v][P * ty];
                    if ((multi >> v) & 1)
                        walk_tile<ARITH, P, P, 1, true, true>(g, u, x0, S, Ls, &acc[0][0]);
                    else if ((clipped >> v) & 1)
                        walk_tile<ARITH, P, P, 1, true>(g, u, x0, S, Ls, &acc[0][0]);
                    else
                        walk_tile<ARITH, P, P, 1, false>(g, u, x0, S, Ls, &acc[0][0]);
                } else {
                    const float u = line_coord(cc, nh), x0 = (float)(rr - nh);
                    const float* Ls = &sLs[v][P * tx];
                    if ((multi >> v) & 1)
                        walk_tile<ARITH, P, 1, P, true, true>(g, u, x0, S, Ls, &acc[0][0]);
                    else if ((clipped >> v) & 1)
                        walk_tile<ARITH, P, 1, P, true>(g, u, x0, S, Ls, &acc[0][0]);
                    else
                        walk_tile<ARITH, P, 1, P, false>(g, u, x0, S, Ls, &acc[0][0]);
                }
                continue;
            }
            const int kind = geom[v0 + v].kind;
            const float* S = &sS[v][0] - sLo[v];
            if (kind == DD_ROWSUM) {
#pragma unroll
                for (int i = 0; i < P; ++i) {
                    const float sv = (rr + i < npix) ? S[rr + i] : 0.0f;
#pragma unroll
                    for (int j = 0; j < P; ++j) acc[i][j] = __fadd_rn(acc[i][j], sv);
                }
            } else if (kind == DD_COLSUM) {
#pragma unroll
                for (int j = 0; j < P; ++j) {
                    const float sv = (cc + j < npix) ? S[cc + j] : 0.0f;
#pragma unroll
                    for (int i = 0; i < P; ++i) acc[i][j] = __fadd_rn(acc[i][j], sv);
                }
            }
        }
    }

    double p1 = 0.0, p2 = 0.0;
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
        for (int j = 0; j < P; ++j) {
            const int r = rr + i, q = cc + j;
            if (r < npix && q < npix) {
                const int64_t o = (int64_t)r * npix + q;
                double q1 = 0.0, q2 = 0.0;
                if (PRE)
                    out[o] = epi_back_v<EPI>(acc[i][j], pre_x[i][j], pre_w[i][j], e, &q1, &q2);
                else if (epi_updates_x(EPI))
                    out[o] = epi_back<EPI>(acc[i][j], out[o], o, z, e, &q1, &q2);
                else
                    out[o] = epi_back<EPI>(acc[i][j], 0.0f, o, z, e, &q1, &q2);
                p1 += q1;
                p2 += q2;
            }
        }
    if (epi_has_partials(EPI) && e.partials)
        block_partials3(0.0, p1, p2,
                        e.partials + ((int64_t)z * e.blocks_per_slice + blk) * 3);
}


__device__ __forceinline__ __amdgpu_buffer_rsrc_t image_rsrc(const float* base, int npix)
{
    // byte size; npix <= 32766 keeps it below 2^32
    const unsigned bytes = (unsigned)npix * (unsigned)npix * 4u;
    return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
}

// image[idx] of one slice; indices outside [0, npix*npix) read 0.
__device__ __forceinline__ float load_px(__amdgpu_buffer_rsrc_t rs, int idx)
{
    // the builtin returns the 32 bits as an integer: reinterpret, do not convert
    return __int_as_float(
        (int)__builtin_amdgcn_raw_buffer_load_b32(rs, (int)((unsigned)idx * 4u), 0, 0));
}

// image[idx .. idx+3] of one slice through the buffer descriptor (out of range: 0).
// idx needs no 16-byte alignment.
__device__ __forceinline__ float4 load_px4(__amdgpu_buffer_rsrc_t rs, int idx)
{
    typedef int int4v __attribute__((ext_vector_type(4)));
    const int4v v = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)((unsigned)idx * 4u), 0, 0);
    return make_float4(__int_as_float(v[0]), __int_as_float(v[1]), __int_as_float(v[2]),
                       __int_as_float(v[3]));
}

// One candidate pixel of a bin [Dlo, Dhi] on a line with offset K: the pixel spans
// [x-K, x+1-K].  Dhc is the bin's right end clipped to the line's L*.  Advances x.
// The first candidate (Rp = x-K, its left end, on entry) can start left of Dlo and gets
// the weight max(min(P_hi, Dhc) - max(P_lo, Dlo), 0).  Every later one gets
// R_k - R_{k-1} with R_k = min(P_hi(k), Dhc), carried in Rp: its left end is the
// previous candidate's right end P_hi(k-1), and where P_hi(k-1) < Dhc that is the same
// subtraction as max(min(P_hi(k), Dhc) - P_hi(k-1), 0), while past the bin's end both
// give +0 (R_k = R_{k-1} = Dhc) -- so no clamp is needed.  A weight of +0 leaves the
// sum unchanged (every candidate value is a finite image value or a zero).
template <int ARITH>
__device__ __forceinline__ float cand_step(bool first, float& x, float& Rp, float K,
                                           float Dlo, float Dhc, float val, float acc)
{
    x = __fadd_rn(x, 1.0f);
    const float R = fminf(__fsub_rn(x, K), Dhc);
    const float w = first ? fmaxf(__fsub_rn(R, fmaxf(Rp, Dlo)), 0.0f) : __fsub_rn(R, Rp);
    Rp = R;
    return accum<ARITH>(w, val, acc);
}

// (index - nh) of the pixel whose span [P_q, P_q+1) holds Dlo on a line with offset K,
// clamped into [0, npix): a floor estimate, then one exact correction against the keys.
__device__ __forceinline__ float first_pixel(float Dlo, float K, int nh, int npix)
{
    // the estimate needs no clamp of its own: far outside the line the correction may
    // be inexact, but the final clamp then lands on the end pixel either way
    float fe = floorf(__fadd_rn(Dlo, K));
    const float fe1 = __fadd_rn(fe, 1.0f);
    const float Pe = __fsub_rn(fe, K);
    const float Pe1 = __fsub_rn(fe1, K);
    // selects, not branches: at most one of the two corrections applies (Pe <= Pe1)
    const float fm1 = __fsub_rn(fe, 1.0f);
    fe = (Dlo >= Pe1) ? fe1 : fe;
    fe = (Dlo < Pe) ? fm1 : fe;
    return __builtin_amdgcn_fmed3f(fe, (float)(-nh), (float)(npix - 1 - nh));
}

// first_pixel with one correction instead of two, for views whose keys all lie below 2^20
// in magnitude (every view with at most 32 candidates per bin and line, the staged and
// the grouped paths: bins narrower than 30.75 pixels and npix <= 32766 bound |D| and |K|
// by 16384 * 30.75 < 2^19; the chunked path for wider views keeps first_pixel).  There every
// rounding of a key or of the estimate is below 1/32, so with q the exact index
// (P_q <= Dlo < P_q+1) and Dlh = fl(Dlo + 1/2), rounded once per bin, floor(fl(Dlh + K)) is
// q or q + 1 and one test against P_fe settles it.
__device__ __forceinline__ float first_pixel_near(float Dlo, float Dlh, float K, int nh, int npix)
{
    float fe = floorf(__fadd_rn(Dlh, K));
    fe = (Dlo < __fsub_rn(fe, K)) ? __fsub_rn(fe, 1.0f) : fe;
    return __builtin_amdgcn_fmed3f(fe, (float)(-nh), (float)(npix - 1 - nh));
}

// Forward projection of unit pixels: one bin over its own lines [i_lo, i_hi], at most NC
// candidate pixels per line (0: g.ncand of them).
template <int ARITH, int NC>
__device__ __forceinline__ float fwd_ones(const DdView& g, const float* __restrict__ ls,
                                          int i_lo, int i_hi, int npix, int nh, float Dlo,
                                          float Dhi, bool last_bin, float acc)
{
    const float xNm1 = (float)(npix - 1 - nh);
    const float Dlh = __fadd_rn(Dlo, 0.5f);
    float u = line_coord(i_lo, nh);
    for (int i = i_lo; i <= i_hi; ++i, u = __fadd_rn(u, 1.0f)) {
        const float K = key_K<ARITH>(g, u);
        float x = NC ? first_pixel_near(Dlo, Dlh, K, nh, npix) : first_pixel(Dlo, K, nh, npix);
        float Dhc = Dhi;
        if (last_bin || Dhi > __fsub_rn(xNm1, K)) Dhc = fminf(Dhi, ls[i]);
        float Rp = __fsub_rn(x, K);
        if (NC) {
#pragma unroll
            for (int k = 0; k < NC; ++k)
                acc = cand_step<ARITH>(k == 0, x, Rp, K, Dlo, Dhc, 1.0f, acc);
        } else {
            for (int k = 0; k < g.ncand; ++k)
                acc = cand_step<ARITH>(k == 0, x, Rp, K, Dlo, Dhc, 1.0f, acc);
        }
    }
    return acc;
}

// Forward projection of one sweep view with wide bins (w = |rinv| pixels, at most NC
// candidates per bin and line, NC = 0: g.ncand of them), along diagonals.
//
// A bin w pixels wide meets only about npix/w lines, and the next bin's lines start
// |1/cos| or |1/sin| (between 1 and sqrt(2) for w >= sqrt(2), towards 1 as w grows) lines
// further on.  So the 64 lanes of a wave, 64 consecutive bins, step together along
// diagonals: in step k lane d takes line L(d) + k, where L(d) is its own first line.  Every
// step then serves all lanes (a block that walks the union of its bins' lines, as the
// staged path does, spends npix/w + 64 line steps where npix/w are needed; staged, the wide
// views alone took 94 us at 64^2 x 45 where the whole forward now takes 18), and the lanes'
// first pixels on their lines agree to within a line's shift.
// Hence candidate j of the wave lies in 64 neighbouring lines at nearly the same place
// along the line: `img` is the orientation in which neighbouring lines are neighbours in
// memory (the transpose of what the staged path reads), and candidate j of the whole wave
// is one nearly contiguous load.  No LDS, no barriers; bounds: vector L1 accesses (one
// 4-byte load per candidate and lane) and the five VALU operations of a candidate.
//
// Lines outside the image (a lane's diagonal before its first or after its last line) load
// nothing and get the right end -1e30, which makes every weight 0.  A weight of 0 makes a NaN of
// an infinity, so the diagonals stay close to the bin's own lines: of the up to GL - 1 lines that
// fill the last group two lie before them and one after (all after, an infinite pixel reached
// bins four lines away; a test of every lane against its own last line cost 1% at 100^2 to
// 256^2), and candidates past g.ncand are not loaded.  Away from the end of the line (q + NC < npix
// for every lane) the candidates need no bounds check and L* does not clip (see dd_fwd_block);
// the last bin of a view always takes the checked form.
template <int ARITH, int NC, int GL>
__device__ __forceinline__ float fwd_diag(const DdView& g, const float* __restrict__ ls,
                                          int npix, int nh, const float* __restrict__ img,
                                          int d, float acc)
{
    constexpr float kNone = -1e30f;
    const __amdgpu_buffer_rsrc_t rs = image_rsrc(img, npix);
    const int dk = min(d, npix - 1);
    const float Dlo = key_D<ARITH>(g, dk - nh);
    const float Dhi = key_D<ARITH>(g, dk + 1 - nh);
    const float Dlh = __fadd_rn(Dlo, 0.5f);
    const bool last_bin = dk == npix - 1;
    // Lines whose pixel span [x0 - K, xN - K] meets [Dlo, Dhi]: K_i = (i - nh + 1/2) t lies
    // between x0 - Dhi and xN - Dlo, a range of (npix + w)/|t| lines; a sixteenth of a line
    // of margin at each end covers every rounding of a key (below 0.01 lines, npix <= 32766).
    const double rt = 1.0 / (double)g.t;
    const double e0 = ((double)(-nh) - (double)Dhi) * rt;
    const double e1 = ((double)(npix - nh) - (double)Dlo) * rt;
    const int L = (int)floor(fmin(e0, e1) + ((double)nh - 0.5625)) + 1;
    const int steps = (int)floor(((double)npix + (double)g.rinv) * fabs(rt) + 0.14) + 1;
    // L is monotonic in the bin: its extremes are in the first and the last lane
    const int La = __builtin_amdgcn_readlane(L, 0), Lb = __builtin_amdgcn_readlane(L, 63);
    const int k1 = min(steps - 1, npix - 1 - min(La, Lb));
    int k0 = max(0, -max(La, Lb));
    k0 -= min(2, (GL - (k1 - k0 + 1) % GL) % GL);   // groups of GL lines, see above
    const int stride = npix * 4;
    if constexpr (NC > 0) {
        for (int k = k0; k <= k1; k += GL) {
            float K[GL], xq[GL], Dhc[GL], v[GL][NC];
            int q[GL], vo[GL];
            bool ok[GL];
            bool edge = last_bin;
#pragma unroll
            for (int l = 0; l < GL; ++l) {
                const int i = L + k + l;
                ok[l] = (unsigned)i < (unsigned)npix;
                K[l] = key_K<ARITH>(g, line_coord(i, nh));
                xq[l] = first_pixel_near(Dlo, Dlh, K[l], nh, npix);
                q[l] = (int)xq[l] + nh;
                edge |= ok[l] && q[l] >= npix - NC;
                vo[l] = ok[l] ? (int)((__umul24(q[l], npix) + (unsigned)i) * 4u) : -1;
            }
            if (!__any(edge)) {
#pragma unroll
                for (int l = 0; l < GL; ++l) {
                    Dhc[l] = ok[l] ? Dhi : kNone;
#pragma unroll
                    for (int j = 0; j < NC; ++j)
                        v[l][j] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(
                            rs, vo[l], j * stride, 0));
                }
            } else {
#pragma unroll
                for (int l = 0; l < GL; ++l) {
                    Dhc[l] = ok[l] ? fminf(Dhi, ls[ok[l] ? L + k + l : 0]) : kNone;
#pragma unroll
                    for (int j = 0; j < NC; ++j)
                        v[l][j] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(
                            rs, ok[l] && q[l] + j < npix ? vo[l] + j * stride : -1, 0, 0));
                }
            }
#pragma unroll
            for (int l = 0; l < GL; ++l) {
                float xk = xq[l], Rp = __fsub_rn(xq[l], K[l]);
#pragma unroll
                for (int j = 0; j < NC; ++j)
                    acc = cand_step<ARITH>(j == 0, xk, Rp, K[l], Dlo, Dhc[l], v[l][j], acc);
            }
        }
    } else {
        constexpr int CH = 16;   // candidates loaded together
        for (int k = k0; k <= k1; ++k) {
            const int i = L + k;
            const bool ok = (unsigned)i < (unsigned)npix;
            const float K = key_K<ARITH>(g, line_coord(i, nh));
            const float x = first_pixel(Dlo, K, nh, npix);
            const int q = (int)x + nh;
            const int vo = ok ? (int)((__umul24(q, npix) + (unsigned)i) * 4u) : -1;
            float Dhc = ok ? Dhi : kNone;
            if (__any(last_bin || (ok && q >= npix - g.ncand)))
                Dhc = ok ? fminf(Dhi, ls[ok ? i : 0]) : kNone;
            float xk = x, Rp = __fsub_rn(x, K);
            for (int j0 = 0; j0 < g.ncand; j0 += CH) {
                float v[CH];
                if (j0 + CH <= g.ncand && !__any(ok && q + j0 + CH > npix)) {
#pragma unroll
                    for (int j = 0; j < CH; ++j)
                        v[j] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(
                            rs, vo, (j0 + j) * stride, 0));
                } else {
                    const int last = min(npix - q, g.ncand) - j0;
#pragma unroll
                    for (int j = 0; j < CH; ++j)
                        v[j] = __int_as_float((int)__builtin_amdgcn_raw_buffer_load_b32(
                            rs, ok && j < last ? vo + (j0 + j) * stride : -1, 0, 0));
                }
#pragma unroll
                for (int j = 0; j < CH; ++j)
                    acc = cand_step<ARITH>(j0 + j == 0, xk, Rp, K, Dlo, Dhc, v[j], acc);
            }
        }
    }
    return acc;
}

// LDS of the staged forward path: 16 floats per thread of the block (64 B bytes for B
// threads, 4 KB per wave), shared by every candidate count.
template <int B>
constexpr int fwd_stage_floats() { return 16 * B; }
constexpr int kFwdStageMaxLines = 8;

// Forward projection of one sweep view with at most NC candidate pixels per bin and line
// (bins narrower than w < NC - 1.25 pixels), for the B bins [bx*B, +B) of a block.
// Lines are processed in chunks of FL: for each line of a chunk the block copies the
// window of W pixels its bins can touch into LDS with 16-byte loads (one contiguous
// row segment per line; the window starts at q0, the first bin's estimated first pixel
// minus 2, rounded down to a multiple of 4), then every thread reads its candidates from
// LDS.  A bin's first candidate lies less than B*w + 6 pixels past q0: less than
// (B-1)*w + 1 + 5 for a bin that starts on the line, and for the last bin up to one bin
// width more where it starts left of the line's first pixel and its first candidate is
// clamped up to that pixel.  With W = (NC-1)*B >= B*w + 6 + NC (for w < NC - 1.25 and B >=
// 4 (NC + 6)) the window holds every candidate of every bin that meets the line.  q0 itself is
// kept in [-(W - NC), npix - 1], which moves it only on lines that every bin of the block misses,
// so that each first candidate, clamped into the line, lies in the window, whatever the bin.
// Lines run over the union of the block's per-bin line ranges; lines that miss a bin add nothing
// to it.  A chunk always runs all its FL lines (straight-line code, so the LDS reads of one line
// hide behind the sums of another): those past the block's last line are zeros with the line end
// kNoLine, which makes every weight 0.  Every thread of the block takes part (inactive threads,
// past the last bin, compute a copy of the last bin and store nothing).
// sImg holds FLOATS floats, sMeta kFwdStageMaxLines entries {byte offset of pixel 0, L*}.
constexpr float kNoLine = -1e30f;

template <int ARITH, int B, int NC, int FLOATS>
__device__ __forceinline__ float fwd_staged(const DdView& g, const float* __restrict__ ls,
                                            int npix, int nh, __amdgpu_buffer_rsrc_t rs,
                                            int bx, int d, float acc, float* sImg,
                                            float2* sMeta)
{
    static_assert(B >= 4 * (NC + 6), "the window holds a block's candidates");
    constexpr int W = (NC - 1) * B;
    constexpr int FL = FLOATS / W < kFwdStageMaxLines ? FLOATS / W : kFwdStageMaxLines;
    constexpr int N4 = FL * (W / 4);          // 16-byte pieces per chunk
    constexpr int PER = (N4 + B - 1) / B;     // pieces per thread
    static_assert(FL >= 1 && W % 4 == 0, "staged window shape");
    const int tid = threadIdx.x;
    const int dk = min(d, npix - 1);
    const float Dlo = key_D<ARITH>(g, dk - nh);
    const float Dhi = key_D<ARITH>(g, dk + 1 - nh);
    const float Dlh = __fadd_rn(Dlo, 0.5f);
    const int d0 = bx * B, d1 = min(d0 + B - 1, npix - 1);
    const float D0lo = key_D<ARITH>(g, d0 - nh);
    const float D1hi = key_D<ARITH>(g, d1 + 1 - nh);
    const float x0 = (float)(-nh), xN = (float)(npix - nh);
    const double rt = 1.0 / (double)g.t;
    double ua = ((double)x0 - (double)D1hi) * rt;
    double ub = ((double)xN - (double)D0lo) * rt;
    if (ua > ub) { const double tmp = ua; ua = ub; ub = tmp; }
    ua = fmin(fmax(ua + nh - 0.5, -4.0), (double)npix + 4.0);
    ub = fmin(fmax(ub + nh - 0.5, -4.0), (double)npix + 4.0);
    const int i_lo = max(0, (int)floor(ua) - 2);
    const int i_hi = min(npix - 1, (int)ceil(ub) + 2);
    const int total = npix * npix;

    float4 v[PER];
    float2 meta;
    // First pixel of the window of line i.
    auto start = [&](int i) {
        const int q = (int)floorf(__fadd_rn(D0lo, key_K<ARITH>(g, line_coord(i, nh)))) + nh - 2;
        return min(max(q, -((W - NC) & ~3)), npix - 1) & ~3;
    };
    // Every load of a chunk is in flight before any is stored.  A window that starts left of
    // the row gets zeros there; past the row's end it holds the next row, never weighted;
    // outside the slice the loads return 0.
    auto load = [&](int c0) {
        // a piece may straddle the slice's end (the last window ends before this index)
        const bool ragged = (npix & 3) && (c0 + FL + 1) * npix + W >= total;
#pragma unroll
        for (int r = 0; r < PER; ++r) {
            const int k = tid + r * B;
            const int l = k / (W / 4), j4 = k - l * (W / 4);
            const int i = c0 + l;
            const int q = start(i) + 4 * j4;
            const int idx = i * npix + q;
            const bool ok = (N4 % B == 0 || k < N4) && i <= i_hi && q >= 0;
            if (!ragged || !ok || idx + 3 < total) {
                v[r] = load_px4(rs, ok ? idx : 0x3fffffff);
            } else {
                v[r].x = load_px(rs, idx);
                v[r].y = load_px(rs, idx + 1);
                v[r].z = load_px(rs, idx + 2);
                v[r].w = load_px(rs, idx + 3);
            }
        }
        const int i = c0 + tid;
        if (tid < FL) {
            meta.x = __int_as_float(4 * (nh - start(i) + tid * W));
            meta.y = i <= i_hi ? ls[i] : kNoLine;
        }
    };
    auto store = [&]() {
#pragma unroll
        for (int r = 0; r < PER; ++r) {
            const int k = tid + r * B;
            if (N4 % B == 0 || k < N4) *(float4*)&sImg[4 * k] = v[r];
        }
        if (tid < FL) sMeta[tid] = meta;
    };

    for (int c0 = i_lo; c0 <= i_hi; c0 += FL) {
        load(c0);
        __syncthreads();  // the previous chunk is consumed
        store();
        __syncthreads();
        float Kp = 0.0f, xp = 0.0f, ep = 0.0f, pv[NC];
#pragma unroll
        for (int l = 0; l <= FL; ++l) {
            float K = 0.0f, x = 0.0f, e = 0.0f, val[NC];
            if (l < FL) {
                K = key_K<ARITH>(g, line_coord(c0 + l, nh));
                x = first_pixel_near(Dlo, Dlh, K, nh, npix);
                const float2 m = sMeta[l];
                e = m.y;
                const float* wp =
                    (const float*)((const char*)sImg + (((int)x << 2) + __float_as_int(m.x)));
#pragma unroll
                for (int k = 0; k < NC; ++k) val[k] = wp[k];
            }
            if (l > 0) {
                // clipping every weight's right end to L* is the exact rule; it changes
                // only the weights that end at the line's dropped segment
                const float Dhc = fminf(Dhi, ep);
                float xk = xp, Rp = __fsub_rn(xp, Kp);
#pragma unroll
                for (int k = 0; k < NC; ++k)
                    acc = cand_step<ARITH>(k == 0, xk, Rp, Kp, Dlo, Dhc, pv[k], acc);
            }
            Kp = K;
            xp = x;
            ep = e;
#pragma unroll
            for (int k = 0; k < NC; ++k) pv[k] = val[k];
        }
    }
    return acc;
}

// How a forward launch takes its views: those with at most fwd_staged_max(path) candidates are
// staged, the others go along diagonals (which path: fwd_path).  Both kinds of views share one
// launch: their waves wait for different units.  (The diagonal ones in a launch of their own: 4967
// us at 2048^2 x 1800 after the staged ones, 4603 beside them on another stream, 4432 so.)
constexpr int fwd_staged_max(int path) { return path == kFwdSmall ? 3 : 6; }

// Forward projection: one thread per (bin, view, slice).
// Lines are image rows for row sweeps and image columns for column sweeps.  Each path reads
// the image or its transpose, whichever makes the lanes of a wave, which hold consecutive
// bins, read consecutive addresses.
// Bins [bx*B, +B) of view `view`, slice z, one per thread; blk indexes the partials.
template <int ARITH, int EPI, bool ONES, int B, int PATH>
__device__ __forceinline__ void dd_fwd_block(const DdView* __restrict__ geom,
                                             const float* __restrict__ lstar, int nang,
                                             int npix, const float* __restrict__ image,
                                             const float* __restrict__ imageT,
                                             float* __restrict__ out, int64_t img_stride,
                                             int64_t sino_stride, int accumulate,
                                             const EpiArgs& e, int bx, int view, int z)
{
    const int d = bx * B + threadIdx.x;
    const bool active = d < npix;
    const DdView g = geom[view];
    image += (int64_t)z * img_stride;
    imageT += (int64_t)z * img_stride;
    const int64_t soff = (int64_t)z * sino_stride;
    const int64_t o = (int64_t)g.row * npix + d;
    const int nh = (int)(npix * 0.5);
    double p0 = 0.0;

    const bool sweep = g.kind == DD_SWEEP_ROWS || g.kind == DD_SWEEP_COLS;
    if (!ONES && sweep) {
        // block-uniform: every thread joins (threads past the last bin compute a copy of
        // it and store nothing); the epilogue inputs are loaded first so that their latency
        // hides behind the sweep
        const EpiFwdIn pre = active ? epi_fwd_load<EPI>(o, soff, z, e) : EpiFwdIn{0.0f, 0.0f};
        float acc = (EPI == EPI_STORE && accumulate && active) ? out[soff + o] : 0.0f;
        const float* ls = lstar + (int64_t)view * npix;
        const int nc = g.ncand;
        constexpr int SMAX = fwd_staged_max(PATH);
        if (nc <= SMAX) {
            constexpr int FLOATS = fwd_stage_floats<B>();
            __shared__ __attribute__((aligned(16))) float sImg[FLOATS];
            __shared__ float2 sMeta[kFwdStageMaxLines];
            const __amdgpu_buffer_rsrc_t rs =
                image_rsrc((g.kind == DD_SWEEP_ROWS) ? image : imageT, npix);
            if (nc <= 3)
                acc = fwd_staged<ARITH, B, 3, FLOATS>(g, ls, npix, nh, rs, bx, d, acc, sImg,
                                                      sMeta);
            else if (SMAX >= 4 && nc == 4)
                acc = fwd_staged<ARITH, B, 4, FLOATS>(g, ls, npix, nh, rs, bx, d, acc, sImg,
                                                      sMeta);
            else if (SMAX >= 5)
                acc = fwd_staged<ARITH, B, 6, FLOATS>(g, ls, npix, nh, rs, bx, d, acc, sImg,
                                                      sMeta);
        } else {
            const float* img = (g.kind == DD_SWEEP_ROWS) ? imageT : image;
#define ITOMO_DIAG(NC, GL) acc = fwd_diag<ARITH, NC, GL>(g, ls, npix, nh, img, d, acc)
            if (SMAX < 4 && nc <= 4) ITOMO_DIAG(4, 4);
            else if (SMAX < 5 && nc <= 5) ITOMO_DIAG(5, 4);
            else if (SMAX < 6 && nc <= 6) ITOMO_DIAG(6, 3);
            else if (nc <= 7) ITOMO_DIAG(7, 2);
            else if (nc <= 8) ITOMO_DIAG(8, 2);
            else if (nc <= 10) ITOMO_DIAG(10, 2);
            else if (nc <= 12) ITOMO_DIAG(12, 2);
            else if (nc <= 16) ITOMO_DIAG(16, 1);
            else if (nc <= 20) ITOMO_DIAG(20, 1);
            else if (nc <= 24) ITOMO_DIAG(24, 1);
            else if (nc <= 32) ITOMO_DIAG(32, 1);
            else ITOMO_DIAG(0, 1);
#undef ITOMO_DIAG
        }
        if (active) out[soff + o] = epi_forward<EPI>(acc, pre, &p0);
    } else if (active) {
        float acc = (EPI == EPI_STORE && accumulate) ? out[soff + o] : 0.0f;
        if (g.kind == DD_ROWSUM) {
            // sum_j img[d][j], in j order, read as column d of the transpose
            const float* p = imageT + d;
            for (int j = 0; j < npix; ++j)
                acc = __fadd_rn(acc, ONES ? 1.0f : p[(int64_t)j * npix]);
        } else if (g.kind == DD_COLSUM) {
            const float* p = image + d;
            for (int j = 0; j < npix; ++j)
                acc = __fadd_rn(acc, ONES ? 1.0f : p[(int64_t)j * npix]);
        } else if (sweep) {   // unit pixels
            const float Dlo = key_D<ARITH>(g, d - nh);
            const float Dhi = key_D<ARITH>(g, d + 1 - nh);
            const float* ls = lstar + (int64_t)view * npix;
            const float x0 = (float)(-nh), xN = (float)(npix - nh);
            // lines whose pixel span [x0 - K, xN - K] can meet [Dlo, Dhi]:
            // x0 - Dhi < K_i < xN - Dlo with K_i ~ (i - nh + 0.5) * t, two lines of margin
            // (margin lines that miss the bin add nothing).
            double ua = ((double)x0 - (double)Dhi) / (double)g.t;
            double ub = ((double)xN - (double)Dlo) / (double)g.t;
            if (ua > ub) { const double tmp = ua; ua = ub; ub = tmp; }
            ua = fmin(fmax(ua + nh - 0.5, -4.0), (double)npix + 4.0);
            ub = fmin(fmax(ub + nh - 0.5, -4.0), (double)npix + 4.0);
            const int i_lo = max(0, (int)floor(ua) - 2);
            const int i_hi = min(npix - 1, (int)ceil(ub) + 2);
            // Lines outside the bin, and candidates past the bin or past the line's end,
            // need no test: the first pixel is clamped into [0, npix), and every weight's
            // right end is clipped to L* <= P[N], so such candidates have R <= L.
            // L* >= min(P[N-1], D[N-1]) on every line, so the clip (and the table read)
            // is needed only where Dhi exceeds that bound: the line's last pixel or the
            // last bin.
            const int nc = g.ncand;
            const bool last = d == npix - 1;
#define ITOMO_ONES(NC) acc = fwd_ones<ARITH, NC>(g, ls, i_lo, i_hi, npix, nh, Dlo, Dhi, last, acc)
            if (nc <= 3) ITOMO_ONES(3);
            else if (nc == 4) ITOMO_ONES(4);
            else if (nc <= 6) ITOMO_ONES(6);
            else if (nc <= 8) ITOMO_ONES(8);
            else if (nc <= 12) ITOMO_ONES(12);
            else if (nc <= 16) ITOMO_ONES(16);
            else ITOMO_ONES(0);
#undef ITOMO_ONES
        }
        out[soff + o] = epi_forward<EPI>(acc, o, soff, z, e, &p0);
    }
    // one FP64 slot per 64-bin chunk of the view (the layout of dd_fwd_slots); a wave
    // past the last bin has no chunk and writes nothing
    const int chunk = bx * (B / 64) + (int)(threadIdx.x >> 6);
    if (epi_has_partials(EPI) && e.partials && chunk * 64 < npix)
        wave_partials3(p0, 0.0, 0.0,
                       e.partials + ((int64_t)z * e.blocks_per_slice +
                                     (int64_t)view * ((npix + 63) / 64) + chunk) * 3);
}

// out[c][r] = in[r][c] for one 32x32 tile of one npix x npix slice, through LDS
// (block 32 x 8 threads).
__device__ __forceinline__ void transpose_tile(const float* __restrict__ in,
                                               float* __restrict__ out, int npix,
                                               int64_t stride, int bx, int by, int z)
{
    __shared__ float tile[32][33];
    in += (int64_t)z * stride;
    out += (int64_t)z * stride;
    const int c0 = bx * 32, r0 = by * 32;
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int r = r0 + k, c = c0 + threadIdx.x;
        if (r < npix && c < npix) tile[k][threadIdx.x] = in[(int64_t)r * npix + c];
    }
    __syncthreads();
    for (int k = threadIdx.y; k < 32; k += 8) {
        const int r = c0 + k, c = r0 + threadIdx.x;  // output row = input column
        if (r < npix && c < npix) out[(int64_t)r * npix + c] = tile[threadIdx.x][k];
    }
}

}  // namespace itomo
