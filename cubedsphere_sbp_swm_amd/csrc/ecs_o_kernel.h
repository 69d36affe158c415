// Device side of the ECS cubic halo on O points, shared by the A-grid entry points (swm_ecs.hip) and
// the C-grid operators (swm_cgrid_ecs.hip).
#pragma once

#include "swm_kernels.h"

namespace swm {

// ---- ECS cubic halo on O points (cell centres of the A grid) ----
// get_ecs_halo / ext_ecs_tile_halo (equiang_cs/ecs_halo_mod.f90:71-166) after the width-8 'full'
// O-point exchange (parallel/exchange_factory_mod.f90:13-28,45-155), which fills the strip beyond
// each panel edge with the edge neighbour's cells and leaves the halo corner squares alone.  Every
// value the procedure writes is a function of the panel and those strips only:
//  - halo row r of an edge at position t along it: 4-point Lagrange interpolation along the
//    neighbour's row at depth r-1 (ecs_ext_halo_1e, :451-475), positions 2..N-1 in row 1 and
//    1..N beyond;
//  - the special points at each cube corner (ecs_halo_1corner, :215-285, placed by
//    ecs_halo_corners_put, :287-334): row 1 at positions 1 and N, the corner-square diagonal and,
//    for hw >= 2, the rest of the 2 x 2 block next to the corner.
// One thread computes one output point from f directly.  Points of the corner squares the
// procedure does not write (only for hw >= 3) are set to NaN.
template <typename T>
struct EcsO {
    using value_type = T;
    const T *f;        // [6][N][N], i fastest
    const T *w;        // [rows][N+4][4]: positions -1..N+2, stencil offsets -1..2
    const int *ind;    // [rows][N+4]: 1-based stencil base
    const int *edge;   // [6][4][8]: neighbour panel, normal axis is x, far side, orientation, vector code
    int N, hw;

    __device__ T at(int p, int i, int j) const { return f[((long long)p * N + j - 1) * N + i - 1]; }
    // exchanged value beyond edge e (0 W, 1 E, 2 S, 3 N) at depth d (0 = first cell row of the
    // neighbour), position t = 1..N along the edge
    __device__ T raw(int p, int e, int d, int t) const {
        const int *ed = edge + (p * 4 + e) * 8;
        const int nidx = ed[2] == 0 ? d : N - 1 - d, tidx = ed[3] > 0 ? t - 1 : N - t;
        const int qi = ed[1] ? nidx : tidx, qj = ed[1] ? tidx : nidx;
        return f[((long long)ed[0] * N + qj) * N + qi];
    }
    // the exchanged array pf(I, J) where one of I, J lies in 1..N
    __device__ T pf(int p, int I, int J) const {
        if (I >= 1 && I <= N && J >= 1 && J <= N) return at(p, I, J);
        if (J < 1) return raw(p, 2, -J, I);
        if (J > N) return raw(p, 3, J - N - 1, I);
        if (I < 1) return raw(p, 0, -I, J);
        return raw(p, 1, I - N - 1, J);
    }
    __device__ T W(int s, int t, int r) const { return w[((r - 1) * (N + 4) + t + 1) * 4 + s + 1]; }
};

// Vector halo on O points (A grid, contravariant components; create_ecs_A_vec_halo_procedure,
// ecs_halo_vec_a_mod.f90:66-192): the exchanged neighbour components (u, v), swapped and negated
// by the panel pair's code (pack_to_buf_vec, parallel/buffer_mod.f90:171-277), times the 2 x 2
// matrix TM of the edge at rows 1..hw (positions ish..ieh) and at rows hw+1..5 near the corners
// (positions ish..2, N-1..ieh); then the scalar procedure on component `comp` (0 u, 1 v).
template <typename T>
struct EcsOVec {
    using value_type = T;
    const T *fu, *fv, *w;
    const int *ind, *edge;
    const T *tm;       // [edge 1..4][tmrows][N][4]
    int N, hw, tmrows, ish, ieh, comp;

    __device__ T at(int p, int i, int j) const {
        const long long o = ((long long)p * N + j - 1) * N + i - 1;
        return comp ? fv[o] : fu[o];
    }
    __device__ T raw(int p, int e, int d, int t) const {
        const int *ed = edge + (p * 4 + e) * 8;
        const int nidx = ed[2] == 0 ? d : N - 1 - d, tidx = ed[3] > 0 ? t - 1 : N - t;
        const int qi = ed[1] ? nidx : tidx, qj = ed[1] ? tidx : nidx;
        const long long o = ((long long)ed[0] * N + qj) * N + qi;
        T zu, zv;
        map_vec(ed[4], fu[o], fv[o], zu, zv);
        const int r = d + 1;
        const bool in = t >= ish && t <= ieh;
        if ((r <= hw && in) || (r > hw && r <= 5 && in && (t <= 2 || t >= N - 1))) {
            const int en = e == 2 ? 1 : e == 3 ? 2 : e == 0 ? 3 : 4;   // the reference's edge number
            const T *m = tm + (((long long)(en - 1) * tmrows + r - 1) * N + t - 1) * 4;
            return comp ? m[2] * zu + m[3] * zv : m[0] * zu + m[1] * zv;
        }
        return comp ? zv : zu;
    }
    __device__ T pf(int p, int I, int J) const {
        if (I >= 1 && I <= N && J >= 1 && J <= N) return at(p, I, J);
        if (J < 1) return raw(p, 2, -J, I);
        if (J > N) return raw(p, 3, J - N - 1, I);
        if (I < 1) return raw(p, 0, -I, J);
        return raw(p, 1, I - N - 1, J);
    }
    __device__ T W(int s, int t, int r) const { return w[((r - 1) * (N + 4) + t + 1) * 4 + s + 1]; }
};

// special value k (0..5) of corner c (0..3: (1,1), (N,1), (N,N), (1,N) sides), ecs_halo_1corner.
// Inlined: a call would make every thread of ecs_o_fill copy its argument struct to scratch
// memory to pass it by reference.
template <typename S>
__device__ __forceinline__ typename S::value_type ecs_o_special(const S &o, int p, int c, int k) {
    using T = typename S::value_type;
    const int N = o.N;
    const int ist = (c == 1 || c == 2) ? N + 1 : 0, idir = (c == 1 || c == 2) ? -1 : 1;
    const int jst = c >= 2 ? N + 1 : 0, jdir = c >= 2 ? -1 : 1;
    auto FC = [&](int a, int b) { return o.pf(p, ist + idir * a, jst + jdir * b); };
    // weights of corner 1; mirrored, w(2:-1:-1, N+2:N-1:-1, :), where the corner is on the right
    auto PW = [&](int s, int t, int r) { return idir == 1 ? o.W(s, t, r) : o.W(1 - s, N + 1 - t, r); };
    const T z0 = PW(0, 1, 1), z1 = PW(1, 1, 1), z2 = PW(2, 1, 1);
    const T zw = PW(-1, 1, 1), zw2 = zw * zw, zw3 = zw2 * zw;
    if (k == 0 || k == 2) {
        const T zx = z0 * FC(0, 1) + z1 * FC(0, 2) + z2 * FC(0, 3);
        const T zy = z0 * FC(1, 0) + z1 * FC(1, -1) + z2 * FC(1, -2);
        const T zz = z0 * FC(1, 1) + z1 * FC(2, 1) + z2 * FC(3, 1);
        if (k == 0) return (zx + zw * zy + zw2 * zz) / (T(1) - zw3);
        const T zfy1 = (zy + zw * zz + zw2 * zx) / (T(1) - zw3);
        const T xx = z0 * FC(1, 0) + z1 * FC(2, 0) + z2 * FC(3, 0);
        const T yy = z0 * FC(0, 1) + z1 * FC(-1, 1) + z2 * FC(-2, 1);
        const T zz2 = z0 * FC(1, 1) + z1 * FC(1, 2) + z2 * FC(1, 3);
        const T zfy2 = (yy + zw * zz2 + zw2 * xx) / (T(1) - zw3);
        const T zff1 = PW(-1, 1, 2) * FC(2, 0) + PW(0, 1, 2) * FC(2, -1) + PW(1, 1, 2) * FC(2, -2) + PW(2, 1, 2) * FC(2, -3);
        const T zff2 = PW(-1, 1, 2) * FC(0, 2) + PW(0, 1, 2) * FC(-1, 2) + PW(1, 1, 2) * FC(-2, 2) + PW(2, 1, 2) * FC(-3, 2);
        return T(0.5) * (PW(-1, 0, 1) * zff1 + PW(0, 0, 1) * zfy1 + PW(1, 0, 1) * FC(0, 1) + PW(2, 0, 1) * FC(0, 2) +
                         PW(-1, 0, 1) * zff2 + PW(0, 0, 1) * zfy2 + PW(1, 0, 1) * FC(1, 0) + PW(2, 0, 1) * FC(2, 0));
    }
    if (k == 1) {
        const T zx = z0 * FC(1, 0) + z1 * FC(2, 0) + z2 * FC(3, 0);
        const T zy = z0 * FC(0, 1) + z1 * FC(-1, 1) + z2 * FC(-2, 1);
        const T zz = z0 * FC(1, 1) + z1 * FC(1, 2) + z2 * FC(1, 3);
        return (zx + zw * zy + zw2 * zz) / (T(1) - zw3);
    }
    const T zff1 = PW(-1, 2, 1) * FC(1, 0) + PW(0, 2, 1) * FC(1, -1) + PW(1, 2, 1) * FC(1, -2) + PW(2, 2, 1) * FC(1, -3);
    const T zff2 = PW(-1, 2, 1) * FC(0, 1) + PW(0, 2, 1) * FC(-1, 1) + PW(1, 2, 1) * FC(-2, 1) + PW(2, 2, 1) * FC(-3, 1);
    if (k == 3) return PW(-1, 0, 2) * zff1 + PW(0, 0, 2) * FC(-1, 1) + PW(1, 0, 2) * FC(-1, 2) + PW(2, 0, 2) * FC(-1, 3);
    if (k == 4) return PW(-1, 0, 2) * zff2 + PW(0, 0, 2) * FC(1, -1) + PW(1, 0, 2) * FC(2, -1) + PW(2, 0, 2) * FC(3, -1);
    const T zff11 = PW(-1, 2, 2) * FC(2, -1) + PW(0, 2, 2) * FC(2, -2) + PW(1, 2, 2) * FC(2, -3) + PW(2, 2, 2) * FC(2, -4);
    const T zff22 = PW(-1, 2, 2) * FC(-1, 2) + PW(0, 2, 2) * FC(-2, 2) + PW(1, 2, 2) * FC(-3, 2) + PW(2, 2, 2) * FC(-4, 2);
    return T(0.5) * (PW(-1, -1, 2) * zff11 + PW(0, -1, 2) * zff1 + PW(1, -1, 2) * FC(-1, 1) + PW(2, -1, 2) * FC(-1, 2) +
                     PW(-1, -1, 2) * zff22 + PW(0, -1, 2) * zff2 + PW(1, -1, 2) * FC(1, -1) + PW(2, -1, 2) * FC(2, -1));
}

// out[(p*L + jj)*L + ii], L = N+2hw, for i, j = ii+1-hw, jj+1-hw
template <typename S>
__global__ void ecs_o_fill(S o, typename S::value_type *__restrict__ out) {
    using T = typename S::value_type;
    const int N = o.N, hw = o.hw, L = N + 2 * hw;
    // 32-bit index arithmetic: 6 L^2 < 2^32 for every panel size the library accepts
    const unsigned LL = (unsigned)L * (unsigned)L;
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 6u * LL) return;
    const int p = (int)(t / LL), r = (int)(t - (unsigned)p * LL);
    const int jj = r / L, ii = r - jj * L;
    const int i = ii + 1 - hw, j = jj + 1 - hw;
    const bool in_i = i >= 1 && i <= N, in_j = j >= 1 && j <= N;
    // corner and special index of a point next to a cube corner (-1 if not special)
    auto special = [&](int &c, int &k) {
        const bool left = i <= 1, bottom = j <= 1;
        c = bottom ? (left ? 0 : 1) : (left ? 3 : 2);
        const int ist = left ? 0 : N + 1, idir = left ? 1 : -1, jst = bottom ? 0 : N + 1, jdir = bottom ? 1 : -1;
        const int ci = idir * (i - ist), cj = jdir * (j - jst);
        k = -1;
        if (ci == 0 && cj == 1) k = 0;
        else if (ci == 1 && cj == 0) k = 1;
        else if (ci == 0 && cj == 0) k = 2;
        else if (hw > 1 && ci == -1 && cj == 0) k = 3;
        else if (hw > 1 && ci == 0 && cj == -1) k = 4;
        else if (hw > 1 && ci == -1 && cj == -1) k = 5;
    };
    T v;
    if (in_i && in_j) {
        v = o.at(p, i, j);
    } else if (in_i || in_j) {
        int e, r, pos;
        if (j < 1) { e = 2; r = 1 - j; pos = i; }
        else if (j > N) { e = 3; r = j - N; pos = i; }
        else if (i < 1) { e = 0; r = 1 - i; pos = j; }
        else { e = 1; r = i - N; pos = j; }
        if (r == 1 && (pos == 1 || pos == N)) {
            int c, k;
            special(c, k);
            v = ecs_o_special(o, p, c, k);
        } else {
            const int b = o.ind[(r - 1) * (N + 4) + pos + 1];
            T s = o.W(-1, pos, r) * o.raw(p, e, r - 1, b - 1);
            s = s + o.W(0, pos, r) * o.raw(p, e, r - 1, b);
            s = s + o.W(1, pos, r) * o.raw(p, e, r - 1, b + 1);
            s = s + o.W(2, pos, r) * o.raw(p, e, r - 1, b + 2);
            v = s;
        }
    } else {
        int c, k;
        special(c, k);
        v = k >= 0 ? ecs_o_special(o, p, c, k) : T(__builtin_nan(""));
    }
    out[t] = v;
}

}  // namespace swm
