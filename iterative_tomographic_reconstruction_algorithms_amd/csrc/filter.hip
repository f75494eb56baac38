// Sinogram filtering for filtered back projection (filters.py:35-113).
//
// The reference zero-pads each row to L = 2*nfreq, nfreq = 2 * 2^ceil(log2 npix), multiplies
// its FFT by a real, even filter array and keeps the first npix samples of the inverse
// FFT.  For outputs 0..npix-1 that is the linear convolution with the real, even taps
// h[k] = (1/L) sum_j H[j] cos(2 pi j k / L) at lags |k| < npix (no wrap-around: L >= 4 npix).
// The taps are computed once on the host in FP64; the GPU convolves each row with them in
// FP64, as a circular convolution of length L = 2^k >= 2 npix - 1 by FFT (fft_device.h).  A row
// is real, so it takes a complex transform of M = L / 2 values, its even samples in the real
// and its odd ones in the imaginary part.  Rows share nothing: a row's bits do not depend on the
// rows beside it.
#include <cmath>
#include <vector>

#include "fft_device.h"
#include "itomo_internal.h"

namespace itomo {

// filters.py:35-76 (dpc = False): half filter for k = 0..nfreq, then mirrored.
static double filter_value(int k, int nfreq, int ftype)
{
    const double f = 2.0 * k / (2.0 * nfreq);   // ramp
    if (k == 0) return 0.0;
    const double w = 2.0 * M_PI * k / (2.0 * nfreq);
    const double d = 1.0;
    switch (ftype) {
    case 1: return f * std::sin(w) / (2.0 * d * 2.0 * d * w);   // shepp-logan
    case 2: return f * std::cos(w) / (2.0 * d * w);             // cosine
    case 3: return f * (0.54 + 0.46 * std::cos(w) / d);        // hamming
    case 4: return f * (1.0 + std::cos(w / d) / 2.0);          // hanning
    default: return f;                                          // ramp
    }
}

constexpr int kFilterMinLog = 6, kFilterMaxLog = 13;   // L up to 8192: 64 KB of LDS

// A row (in LDS: out may be where it came from) convolved directly, the way the sum is written
// down: for rows with an infinity or a NaN, whose effect a transform would spread over the whole
// row.
__device__ void conv_row(const float* in, float* out, const double* __restrict__ taps, int npix,
                         int tid, int nt)
{
    for (int n = tid; n < npix; n += nt) {
        double acc = 0.0;
        for (int m = 0; m < npix; ++m) {
            const int lag = n >= m ? n - m : m - n;
            acc = fma((double)in[m], taps[lag], acc);
        }
        out[n] = (float)acc;
    }
}

// Blocks take rows in turn; each transforms the taps once.  A row is read whole before any of it
// is written, so in and out may be the same array.  Bound by LDS: 2 (k/2 + 1) passes of
// 32 bytes per value and transform.  One output costs about 10 k FP64 operations instead of
// 2 npix (3600 rows of 1024: 59 us; a direct sum over LDS 602).  The error of an output
// is FP64 rounding of the norm of its own row, below 1e-13 of the sum of the terms' sizes.
//
// With Z the transform of the M complex values, E_k = (Z_k + conj Z_M-k) / 2 and
// O_k = (Z_k - conj Z_M-k) / 2i are those of the even and the odd samples, and the row's own
// transform is X_k = E_k + w_k O_k, X_k+M = E_k - w_k O_k, w_k = exp(-2 pi i k / L).  Times the
// taps' spectrum (real, for the taps are real and even; H_k+M = H_M-k) and taken apart again,
// with s = (H_k + H_M-k) / 2 and d = (H_k - H_M-k) / 2:
//   E'_k = s E_k + d w_k O_k,   O'_k = s O_k + d conj(w_k) E_k.
// The taps' own E and O give s = Re E_k and d = Re(w_k O_k).
template <int LOGL>
__global__ void __launch_bounds__((fft_threads<LOGL - 1>()))
filter_rows_kernel(const float* in, float* out, const double* __restrict__ taps, int nrows,
                   int npix)
{
    constexpr int L = 1 << LOGL, M = L / 2, T = fft_threads<LOGL - 1>();
    constexpr int E = (L + T - 1) / T;          // samples per thread
    constexpr int P = M / 2 / T + 1;            // pairs (k, M - k), k = 0 .. M / 2, per thread
    constexpr int NA = L / 64;
    __shared__ double2 buf[M];
    __shared__ double2 sA[NA], sB[64];          // exp(-2 pi i 64 a / L), exp(-2 pi i b / L)
    double* const re = (double*)buf;            // re[n]: sample n
    const int tid = threadIdx.x;
    for (int q = tid; q < NA + 64; q += T) {
        const int k = q < NA ? 64 * q : q - NA;
        double2 w;
        sincospi(-2.0 * k / L, &w.y, &w.x);
        if (q < NA) sA[q] = w; else sB[q - NA] = w;
    }
    auto twl = [&](int q) { return c_mul(sA[q >> 6], sB[q & 63]); };
    auto tw = [&](int q) { return twl(2 * q); };
    // E_k and O_k of the transform in buf
    auto split = [&](int k, double2& ek, double2& ok) {
        const double2 a = buf[k], b = buf[(M - k) & (M - 1)];
        ek = make_double2(0.5 * (a.x + b.x), 0.5 * (a.y - b.y));
        ok = make_double2(0.5 * (a.y + b.y), 0.5 * (b.x - a.x));
    };
    // the spectrum of the even extension of the taps, 1/M folded in
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = tid + e * T, lag = min(i, L - i);
        if (i < L) re[i] = lag < npix ? taps[lag] : 0.0;
    }
    __syncthreads();
    fft_lds<LOGL - 1, T>(buf, tid, 1, tw);
    double hs[P], hd[P];
#pragma unroll
    for (int e = 0; e < P; ++e) {
        const int k = tid + e * T;
        hs[e] = hd[e] = 0.0;
        if (k <= M / 2) {
            double2 ek, ok;
            split(k, ek, ok);
            hs[e] = ek.x * (1.0 / M);
            hd[e] = c_mul(twl(k), ok).x * (1.0 / M);
        }
    }
    for (int row = blockIdx.x; row < nrows; row += gridDim.x) {
        const float* r = in + (int64_t)row * npix;
        float* o = out + (int64_t)row * npix;
        float x[E];
        bool finite = true;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = tid + e * T;
            x[e] = i < npix ? r[i] : 0.0f;
            finite = finite && isfinite(x[e]);
        }
        // also: the last row's (or the taps') buffer is consumed
        if (__syncthreads_or(!finite)) {
            float* const row_in = (float*)buf;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = tid + e * T;
                if (i < npix) row_in[i] = x[e];
            }
            __syncthreads();
            conv_row(row_in, o, taps, npix, tid, T);
            continue;
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = tid + e * T;
            if (i < L) re[i] = x[e];
        }
        __syncthreads();
        fft_lds<LOGL - 1, T>(buf, tid, 1, tw);
        // the inverse transform is the forward one with the parts exchanged; a pair (k, M - k)
        // is read and written by one thread
#pragma unroll
        for (int e = 0; e < P; ++e) {
            const int k = tid + e * T;
            if (k <= M / 2) {
                double2 ek, ok, w = twl(k);
                split(k, ek, ok);
                const double2 wo = c_mul(w, ok);
                w.y = -w.y;
                const double2 we = c_mul(w, ek);
                const double2 en = make_double2(hs[e] * ek.x + hd[e] * wo.x,
                                                hs[e] * ek.y + hd[e] * wo.y);
                const double2 on = make_double2(hs[e] * ok.x + hd[e] * we.x,
                                                hs[e] * ok.y + hd[e] * we.y);
                buf[(M - k) & (M - 1)] = make_double2(on.x - en.y, en.x + on.y);
                buf[k] = make_double2(en.y + on.x, en.x - on.y);
            }
        }
        __syncthreads();
        fft_lds<LOGL - 1, T>(buf, tid, 1, tw);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = tid + e * T;
            if (i < npix) o[i] = (float)re[i ^ 1];
        }
    }
}

template <int LOGL>
static void launch_filter(const float* in, float* out, int nrows, int npix, const double* taps,
                          hipStream_t st)
{
    if constexpr (LOGL <= kFilterMaxLog) {
        if (LOGL == kFilterMaxLog || (1 << LOGL) >= 2 * npix - 1) {
            // as many blocks as the LDS of 256 compute units holds, at least one per unit
            constexpr int lds = (8 << LOGL) + 16 * ((1 << LOGL) / 64 + 64);
            constexpr int T = fft_threads<LOGL - 1>();
            constexpr int fit = 163840 / lds < 2048 / T ? 163840 / lds : 2048 / T;
            const int most = 256 * fit;
            filter_rows_kernel<LOGL><<<nrows < most ? nrows : most, T, 0, st>>>(in, out, taps,
                                                                             nrows, npix);
        } else {
            launch_filter<LOGL + 1>(in, out, nrows, npix, taps, st);
        }
    }
}

}  // namespace itomo

using namespace itomo;

extern "C" {

int itomo_filter_taps(int npix, int ftype, double* taps_host)
{
    if (npix < 1 || npix > 4096 || !taps_host || ftype < 0 || ftype > 5)
        return set_error(ITOMO_EINVAL, "filter_taps: bad argument");
    int p2 = 1;
    while (p2 < npix) p2 <<= 1;
    const int nfreq = 2 * p2, L = 2 * nfreq;
    std::vector<double> H(L);
    for (int j = 0; j < L; ++j) {
        const int k = j <= nfreq ? j : L - j;
        H[j] = ftype == 5 ? 1.0 : filter_value(k, nfreq, ftype);   // 5: 'none'
    }
    for (int k = 0; k < npix; ++k) {
        double s = 0.0;
        for (int j = 0; j < L; ++j)
            s += H[j] * std::cos(2.0 * M_PI * (double)((int64_t)j * k % L) / L);
        taps_host[k] = s / L;
    }
    return ITOMO_OK;
}

int itomo_filter_rows(const float* in, float* out, int nrows, int npix, const double* taps,
                      void* stream)
{
    if (!in || !out || !taps || nrows < 1 || npix < 1 || npix > 4096)
        return set_error(ITOMO_EINVAL, "filter_rows: bad argument");
    launch_filter<kFilterMinLog>(in, out, nrows, npix, taps, (hipStream_t)stream);
    return check_hip(hipGetLastError(), "filter_rows launch");
}

}  // extern "C"
