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

// Sums of the per-block partials (value-major, nblocks each: K pairs (sum, compensation), min, max)
// into out = {K sums, min, max}: one block, two waves to each of the K + 2 values, every lane over each
// 128th partial with eight loads in flight, then the lanes by shuffles and the two waves through LDS,
// compensated additions throughout.  One CU's units and the length of a wave's chain are the time: 4.7 us for
// the 1024 partials of swm_diagnostics, 9.7 us with the values of a block side by side (each lane its own
// line), 11.4 us with every thread on all values of a partial, 371 us with one thread walking them.
// swm_diagnostics at C384 takes 56 us, 424 with that one thread.
constexpr int FINAL_THREADS = 1024;

template <int K>
__device__ __forceinline__ void sum_partials(const double *__restrict__ part, long long nblocks,
                                             double *__restrict__ out) {
    constexpr int PER = 2, LOADS = 8;   // waves per value, loads in flight
    static_assert((K + 2) * PER * 64 <= FINAL_THREADS, "two waves per value");
    __shared__ double sh[K + 2][PER][2];
    const int t = threadIdx.x, lane = t % 64, wave = __builtin_amdgcn_readfirstlane(t / 64);
    const int q = wave / PER, w = wave % PER;   // q < K: sum q, K: min, K + 1: max
    double s = q == K ? 1e300 : q == K + 1 ? -1e300 : 0.0, c = 0.0;
    auto add = [&](double x, double xc) {
        if (q < K) {
            neu_add(s, c, x);
            c += xc;
        } else {
            s = q == K ? fmin(s, x) : fmax(s, x);
        }
    };
    if (q < K + 2) {
        const double *p = part + (q <= K ? 2 * q : 2 * K + 1) * nblocks;
        for (long long b = w * 64 + lane; b < nblocks; b += 64 * PER * LOADS) {
            double x[LOADS], xc[LOADS];
#pragma unroll
            for (int k = 0; k < LOADS; ++k) {
                const long long i = b + 64 * PER * k;
                x[k] = i < nblocks ? p[i] : 0.0;
                xc[k] = q < K && i < nblocks ? p[nblocks + i] : 0.0;
            }
#pragma unroll
            for (int k = 0; k < LOADS; ++k)
                if (b + 64 * PER * k < nblocks) add(x[k], xc[k]);
        }
        for (int off = 32; off > 0; off >>= 1) {
            const double x = __shfl_down(s, off, 64), xc = __shfl_down(c, off, 64);
            add(x, xc);
        }
        if (lane == 0) {
            sh[q][w][0] = s;
            sh[q][w][1] = c;
        }
    }
    __syncthreads();
    if (q >= K + 2 || w != 0 || lane != 0) return;
    add(sh[q][1][0], sh[q][1][1]);
    out[q] = q < K ? s + c : s;
}

}  // namespace swm
