// Sinogram filtering for filtered back projection (filters.py:35-113).
//
// The reference zero-pads each row to L = 2*nfreq, nfreq = 2 * 2^ceil(log2 npix), multiplies
// its FFT by a real, even filter array and keeps the first npix samples of the inverse
// FFT.  For outputs 0..npix-1 that is the linear convolution with the real, even taps
// h[k] = (1/L) sum_j H[j] cos(2 pi j k / L) at lags |k| < npix (no wrap-around: L >= 4 npix).
// The taps are computed once on the host in FP64; the GPU convolves each row with them in
// FP64, as a circular convolution of length L = 2^k >= 2 npix - 1 by FFT (fft_device.h).  The
// taps' spectrum is real (they are real and even), so two rows ride in one complex transform,
// one in the real and one in the imaginary part, and neither reaches the other's result.
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

constexpr int kFilterMinLog = 6, kFilterMaxLog = 13;   // L up to 8192: 128 KB of LDS

// Row r convolved directly, the way the sum is written down: for rows with an infinity or a
// NaN, whose effect a transform would spread over the whole row (and its partner).
__device__ void conv_row(const float* __restrict__ in, float* __restrict__ out,
                         const double* __restrict__ taps, int npix, int tid, int nt)
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

// Blocks take pairs of rows in turn; each transforms the taps once.  Bound by LDS: 2 (k/2 + 1)
// passes of 32 bytes per value and transform.  One output costs about 10 k FP64 operations
// instead of 2 npix (a direct sum over LDS took 687 us for 3600 rows of 1024, this 74).  The error stays at FP64 rounding of the row's norm: rows whose largest
// values differ by more than 2^20 (a zero row beside another included) go through on their own.
template <int LOGL>
__global__ void __launch_bounds__((fft_threads<LOGL>()))
filter_rows_kernel(const float* __restrict__ in, float* __restrict__ out,
                   const double* __restrict__ taps, int nrows, int npix)
{
    constexpr int L = 1 << LOGL, T = fft_threads<LOGL>(), E = (L + T - 1) / T;
    constexpr int NA = L / 64 > 0 ? L / 64 : 1;
    __shared__ double2 buf[L];
    __shared__ double2 sA[NA], sB[64];      // exp(-2 pi i 64 a / L), exp(-2 pi i b / L)
    __shared__ float sMax[2][T / 64];
    const int tid = threadIdx.x;
    for (int q = tid; q < NA + 64; q += T) {
        const int k = q < NA ? 64 * q : q - NA;
        double2 w;
        sincospi(-2.0 * k / L, &w.y, &w.x);
        if (q < NA) sA[q] = w; else sB[q - NA] = w;
    }
    auto tw = [&](int q) { return c_mul(sA[q >> 6], sB[q & 63]); };
    // the spectrum of the even extension of the taps, 1/L folded in
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = tid + e * T, lag = min(i, L - i);
        if (i < L) buf[i] = make_double2(lag < npix ? taps[lag] : 0.0, 0.0);
    }
    __syncthreads();
    fft_lds<LOGL, T>(buf, tid, 1, tw);
    double H[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int i = tid + e * T;
        H[e] = i < L ? buf[i].x * (1.0 / L) : 0.0;
    }
    const int pairs = (nrows + 1) / 2;
    for (int p = blockIdx.x; p < pairs; p += gridDim.x) {
        const float* r0 = in + (int64_t)(2 * p) * npix;
        const bool two = 2 * p + 1 < nrows;
        float x[E], y[E], mx = 0.0f, my = 0.0f;
        bool finite = true;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = tid + e * T;
            x[e] = i < npix ? r0[i] : 0.0f;
            y[e] = two && i < npix ? r0[npix + i] : 0.0f;
            mx = fmaxf(mx, fabsf(x[e]));
            my = fmaxf(my, fabsf(y[e]));
            finite = finite && isfinite(x[e]) && isfinite(y[e]);
        }
        if (!finite) mx = INFINITY;
        for (int off = 32; off > 0; off >>= 1) {
            mx = fmaxf(mx, __shfl_xor(mx, off, 64));
            my = fmaxf(my, __shfl_xor(my, off, 64));
        }
        __syncthreads();   // the last pair's (or the taps') buffer is consumed
        if ((tid & 63) == 0) {
            sMax[0][tid >> 6] = mx;
            sMax[1][tid >> 6] = my;
        }
        __syncthreads();
        for (int w = 0; w < T / 64; ++w) {
            mx = fmaxf(mx, sMax[0][w]);
            my = fmaxf(my, sMax[1][w]);
        }
        float* o0 = out + (int64_t)(2 * p) * npix;
        if (mx == INFINITY) {
            conv_row(r0, o0, taps, npix, tid, T);
            if (two) conv_row(r0 + npix, o0 + npix, taps, npix, tid, T);
            continue;
        }
        const bool apart = fmaxf(mx, my) * 9.5367431640625e-7f > fminf(mx, my);   // 2^-20
        for (int part = 0; part < (apart && two ? 2 : 1); ++part) {
            if (part) __syncthreads();
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = tid + e * T;
                const float re = part ? 0.0f : x[e], im = part || !apart ? y[e] : 0.0f;
                if (i < L) buf[i] = make_double2(re, im);
            }
            __syncthreads();
            fft_lds<LOGL, T>(buf, tid, 1, tw);
            // the inverse transform is the forward one with the parts exchanged
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = tid + e * T;
                if (i < L) buf[i] = make_double2(buf[i].y * H[e], buf[i].x * H[e]);
            }
            __syncthreads();
            fft_lds<LOGL, T>(buf, tid, 1, tw);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = tid + e * T;
                if (i < npix) {
                    if (!part) o0[i] = (float)buf[i].y;
                    if (two && (part || !apart)) o0[npix + i] = (float)buf[i].x;
                }
            }
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
            constexpr int lds = (16 << LOGL) + 16 * ((1 << LOGL) / 64 + 64) + 128;
            constexpr int T = fft_threads<LOGL>();
            constexpr int fit = 163840 / lds < 2048 / T ? 163840 / lds : 2048 / T;
            const int pairs = (nrows + 1) / 2, most = 256 * fit;
            filter_rows_kernel<LOGL><<<pairs < most ? pairs : most, T, 0, st>>>(in, out, taps,
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
