// Compensated sums of the diagnostics (both grids).
#pragma once

#include <hip/hip_runtime.h>

namespace swm {

__device__ __forceinline__ void neu_add(double &s, double &c, double x) {
    const double t = s + x;
    if (fabs(s) >= fabs(x))
        c += (s - t) + x;
    else
        c += (x - t) + s;
    s = t;
}

// Sums of the per-block partials (STRIDE doubles per block: K pairs (sum, compensation), min, max)
// into out = {K sums, min, max}: one block, each thread over every 1024th partial, then the waves'
// lanes by shuffles and the 16 waves through LDS, compensated additions throughout.  One thread
// walking the partials alone is a chain of dependent loads and additions: 371 us for the 1024 of
// swm_diagnostics (72 us for the 216 of a C-grid C90 state).  With this block the whole call at
// C384 takes 64 us instead of 424 us.
constexpr int FINAL_THREADS = 1024;

template <int K>
__device__ __forceinline__ void lanes_combine(double (&s)[K], double (&c)[K], double &lo, double &hi, int width) {
    for (int off = width / 2; off > 0; off >>= 1) {
#pragma unroll
        for (int q = 0; q < K; ++q) {
            const double s2 = __shfl_down(s[q], off, 64), c2 = __shfl_down(c[q], off, 64);
            neu_add(s[q], c[q], s2);
            c[q] += c2;
        }
        lo = fmin(lo, __shfl_down(lo, off, 64));
        hi = fmax(hi, __shfl_down(hi, off, 64));
    }
}

template <int K, int STRIDE>
__device__ __forceinline__ void sum_partials(const double *__restrict__ part, long long nblocks,
                                             double *__restrict__ out) {
    constexpr int NWAVES = FINAL_THREADS / 64;
    __shared__ double sh[NWAVES][2 * K + 2];
    const int t = threadIdx.x, lane = t % 64, wave = t / 64;
    double s[K], c[K], lo = 1e300, hi = -1e300;
#pragma unroll
    for (int q = 0; q < K; ++q) s[q] = c[q] = 0.0;
    for (long long b = t; b < nblocks; b += FINAL_THREADS) {
        const double *p = part + b * STRIDE;
#pragma unroll
        for (int q = 0; q < K; ++q) {
            neu_add(s[q], c[q], p[2 * q]);
            c[q] += p[2 * q + 1];
        }
        lo = fmin(lo, p[2 * K]);
        hi = fmax(hi, p[2 * K + 1]);
    }
    lanes_combine<K>(s, c, lo, hi, 64);
    if (lane == 0) {
#pragma unroll
        for (int q = 0; q < K; ++q) {
            sh[wave][2 * q] = s[q];
            sh[wave][2 * q + 1] = c[q];
        }
        sh[wave][2 * K] = lo;
        sh[wave][2 * K + 1] = hi;
    }
    __syncthreads();
    if (wave != 0) return;
    const int w = lane % NWAVES;
#pragma unroll
    for (int q = 0; q < K; ++q) {
        s[q] = sh[w][2 * q];
        c[q] = sh[w][2 * q + 1];
    }
    lo = sh[w][2 * K];
    hi = sh[w][2 * K + 1];
    lanes_combine<K>(s, c, lo, hi, NWAVES);
    if (lane != 0) return;
#pragma unroll
    for (int q = 0; q < K; ++q) out[q] = s[q] + c[q];
    out[K] = lo;
    out[K + 1] = hi;
}

}  // namespace swm
