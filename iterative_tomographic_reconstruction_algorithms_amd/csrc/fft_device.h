// Power-of-two complex FFTs in LDS, shared by the sinogram filter (FP64) and the gridding
// pair (FP32): Stockham passes of radix 4 (the last one radix 2 for odd powers), natural
// order in and out.  A pass keeps its values in registers between reading and writing the one
// LDS buffer, so a transform of L values needs L values of LDS, not two buffers of them.
#pragma once

#include <hip/hip_runtime.h>

namespace itomo {

template <typename V>
__device__ __forceinline__ V c_mul(V a, V b)
{
    V r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}
template <typename V>
__device__ __forceinline__ V c_add(V a, V b)
{
    V r;
    r.x = a.x + b.x;
    r.y = a.y + b.y;
    return r;
}
template <typename V>
__device__ __forceinline__ V c_sub(V a, V b)
{
    V r;
    r.x = a.x - b.x;
    r.y = a.y - b.y;
    return r;
}

// Threads per transform of 2^LOGL values: 8 values per thread (16 took 285 registers in FP64,
// one wave per SIMD), one wave at least, 1024 threads at most (2^13 values).
template <int LOGL>
constexpr int fft_threads()
{
    return (1 << LOGL) / 8 < 64 ? 64 : (1 << LOGL) / 8;
}

// In-place transform of buf[0 .. 2^LOGL) by T threads (tid = 0 .. T-1), W = exp(-2 pi i sg / L)
// with sg = +1 or -1; tw(q) returns exp(-2 pi i sg q / L).  Every thread of the block calls
// it (the barriers are the block's); buf holds its input behind a barrier, and on return its
// output.
template <int LOGL, int T, typename V, typename TW>
__device__ __forceinline__ void fft_lds(V* buf, int tid, int sg, TW tw)
{
    constexpr int L = 1 << LOGL, E4 = (L / 4 + T - 1) / T, E2 = (L / 2 + T - 1) / T;
    int m = 1;
#pragma unroll 1
    for (int pass = 0; pass < LOGL / 2; ++pass, m *= 4) {
        V v[E4][4];
#pragma unroll
        for (int e = 0; e < E4; ++e) {
            const int j = tid + e * T;
            if (L / 4 % T && j >= L / 4) continue;
            V a[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) a[t] = buf[j + t * (L / 4)];
            const int k = j & (m - 1);
            if (k > 0) {
                const int q = k * (L / (4 * m));
#pragma unroll
                for (int t = 1; t < 4; ++t) a[t] = c_mul(a[t], tw(t * q));
            }
            const V s02 = c_add(a[0], a[2]), d02 = c_sub(a[0], a[2]);
            const V s13 = c_add(a[1], a[3]), d = c_sub(a[1], a[3]);
            V d13;   // -i sg d
            d13.x = sg > 0 ? d.y : -d.y;
            d13.y = sg > 0 ? -d.x : d.x;
            v[e][0] = c_add(s02, s13);
            v[e][1] = c_add(d02, d13);
            v[e][2] = c_sub(s02, s13);
            v[e][3] = c_sub(d02, d13);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E4; ++e) {
            const int j = tid + e * T;
            if (L / 4 % T && j >= L / 4) continue;
            const int k = j & (m - 1), base = (j - k) * 4 + k;
#pragma unroll
            for (int t = 0; t < 4; ++t) buf[base + t * m] = v[e][t];
        }
        __syncthreads();
    }
    if constexpr (LOGL & 1) {
        V v[E2][2];
#pragma unroll
        for (int e = 0; e < E2; ++e) {
            const int j = tid + e * T;
            if (L / 2 % T && j >= L / 2) continue;
            const V a = buf[j];
            V b = buf[j + L / 2];
            if (j > 0) b = c_mul(b, tw(j));   // m = L / 2, so k = j
            v[e][0] = c_add(a, b);
            v[e][1] = c_sub(a, b);
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E2; ++e) {
            const int j = tid + e * T;
            if (L / 2 % T && j >= L / 2) continue;
            buf[j] = v[e][0];
            buf[j + L / 2] = v[e][1];
        }
        __syncthreads();
    }
}

}  // namespace itomo
