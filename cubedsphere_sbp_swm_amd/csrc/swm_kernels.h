// Device kernels of the Ah-grid vector-invariant shallow-water step (gfx950).
//
// One launch per RK stage evaluates the whole right-hand side of
// operator_swm_t%apply (models/shallow_water/operator/operator_swm_mod.f90:61-113) for a
// tile of points and applies the RK4 stage update (time_schemes/rk4_mod.f90:20-42):
//   * the five stencil inputs K = (u.ut+v.vt)/2 + g h + g hs, J*hu, J*hv, J*(v/J), J*(-u/J)
//     are formed once per point in LDS from the state and the metric;
//   * SBP derivative rows (interior stencil or boundary closure) are applied along x and y;
//     the tiles compute every point off the panel edges;
//   * blocks of their own in the same launch compute the panel-edge points: they load both
//     panels' points along a segment of a shared edge (depth 0 .. closure width) into LDS,
//     evaluate both one-sided derivative rows at the shared points, and combine them with
//     the reference's scalar and covariant-vector edge averaging
//     (halo_Ah_scalar_sync_mod.f90:52-93, ecs_Ah_vec_sync_mod.f90:77-124) -- this replaces
//     the MPI halo exchange;
//   * the Coriolis term, tendencies and the RK stage combination finish in registers.
// FP64 builds use -ffp-contract=off and the reference's operation order, so results agree
// bit for bit with an FP64 CPU evaluation of the same algorithm.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <utility>

#include "sbp_tables.h"

namespace swm {

// ----------------------------------------------------------------------------------------
// Geometry and per-launch arguments
template <typename T>
struct DevGeo {
    const T *J, *Qi11, *Qi12, *Qi22, *f;   // [panel][j][i], row pitch `pitch`
    // panel stride of J, Qi11, Qi12, Qi22 in elements: n*pitch, or 0 where every panel holds the
    // same values (the ECS metric depends on alpha, beta only) and panel 0's copy serves all six
    long long mps;
    const T *qb, *qt, *ql, *qr;            // covariant sync weights, n values each
    const int *einfo;                      // per (panel, edge): q, nu_is_x, tnu, a_base, s, code
    const double *tanA;                    // tan(alpha_i), i = 0..n-1 (metric evaluated on the fly)
    int n, pitch;
    long long fs;                          // elements per field (6*n*pitch)
    T hxs;                                 // hx*scale
    T hx, scale, grav;
};

enum StageMode : int {
    MODE_RHS = 0,     // out = RHS(y)                               (also the first stage of a step: out is k1)
    MODE_STAGE1 = 1,  // out = y + cy*k ; acc = y + cacc*k          (y is the step's v0)
    MODE_STAGE23 = 2, // out = v0 + cy*k ; acc = acc + cacc*k
    MODE_STAGE4 = 3,  // out = acc + cy*k                           (out is v0)
    MODE_CURL = 4,    // out(h plane) = synced relative vorticity of y
    MODE_SLOPE2 = 5,  // out = RHS(y + ck*kin)                      (y is v0, kin k1, out k2)
    MODE_SLOPE3 = 6   // k = RHS(y + ck*kin): out = y + cy*k ; acc = ((y + ck1*acc) + cacc*kin) + cacc*k
                      //                                            (y is v0, kin k2, acc holds k1 on entry)
};
// The stages of a step, rk4_mod.f90:28-40.  Steps of large grids run RHS, SLOPE2, SLOPE3, STAGE4: stages 1 and 2
// write the slope only, 39 field passes a step.  Small grids, ensembles and the adjoint's tape, which wants the
// stage states themselves, run STAGE1, STAGE23, STAGE23, STAGE4, which write them and the sum, 48 passes.  Both form
// every value with the same operations.
SWM_HD constexpr bool mode_slope(int mode) { return mode == MODE_SLOPE2 || mode == MODE_SLOPE3; }

template <typename T>
struct StageArgs {
    const T *y;    // input state: h at y, u at y+fs, v at y+2fs
    T *out;
    const T *v0;
    T *acc;
    const T *hs;   // orography, may be null
    T cy, cacc;
    T *zeta;       // optional: the synced relative vorticity of y is also written here
    const T *kin;  // slope of the previous stage (MODE_SLOPE2, MODE_SLOPE3)
    T ck, ck1;
};

// Tile shapes (columns x rows of points, one thread per point) of the stage kernels: 64 x 8,
// 32 x 16, 16 x 32 (512 threads) and 32 x 8 (256 threads).  tile_width(ty) is the 512-thread
// shape of `ty` rows.
SWM_HD constexpr int tile_width(int ty) { return 512 / ty; }
SWM_HD constexpr bool tile_shape_ok(int tx, int ty) {
    return (tx == 64 && ty == 8) || (tx == 32 && ty == 16) || (tx == 16 && ty == 32) || (tx == 32 && ty == 8);
}
// The tiles cover the points 1 .. n-2 of a panel line (the edge segments own 0 and n-1):
// tiles_along(n, t) tiles of t points, the b-th starting at point 1 + b*t.
SWM_HD constexpr int tiles_along(int n, int t) { return (n - 2 + t - 1) / t; }

// The panel-edge points are computed by edge segments of consecutive points: per panel the
// x-edges (i = 0 and i = n-1, positions j = 0..n-1, cube corners included) and the y-edges (j = 0
// and j = n-1, positions i = 1..n-2).  A segment and the REACH points its tangential rows read on
// either side fill the 64 lanes of a wave.
SWM_HD constexpr int edge_seg_len(int reach) { return 64 - 2 * reach; }
SWM_HD constexpr int edge_segs_x(int n, int reach) { return (n + edge_seg_len(reach) - 1) / edge_seg_len(reach); }
SWM_HD constexpr int edge_segs_y(int n, int reach) { return (n - 2 + edge_seg_len(reach) - 1) / edge_seg_len(reach); }
SWM_HD constexpr int edge_segs(int n, int reach) { return 6 * 2 * (edge_segs_x(n, reach) + edge_segs_y(n, reach)); }

template <typename T>
struct EnsMember {
    DevGeo<T> g;
    StageArgs<T> a;
};

// ----------------------------------------------------------------------------------------
// Pointwise stencil inputs of one point (co2contra_colocated_mod.f90:55-56,
// massflux_colocated_mod.f90:26-27, KE_colocated_mod.f90:44, operator_swm_mod.f90:85,
// div_ah_sbp_mod.f90:80-91, curl_div_based_mod.f90:58-59).
// Here and in all kernels a quotient is a plain division, correctly rounded over the whole range.  Quotients of one
// denominator by a shared, refined reciprocal take less than half the instructions (C384 step alone 79.7 us against 82.7,
// with three contexts at work 79.7 against 80.5; ensemble step 199 against 206), but are not the same where
// the denominator, the quotient or its residual is subnormal.
template <typename T>
struct Derived {
    T K, Gxd, Gyd, Gxc, Gyc;
    T hu, hv;  // h*ut, h*vt (kept in registers for the point's own output)
};

template <typename T>
__device__ __forceinline__ Derived<T> make_derived(T h, T u, T v, T J, T q11, T q12, T q22, T hsv, T grav) {
    Derived<T> d;
    const T ut = q11 * u + q12 * v;
    const T vt = q12 * u + q22 * v;
    const T hu = h * ut;
    const T hv = h * vt;
    T K = (u * ut + v * vt) / T(2);
    K = K + grav * h + grav * hsv;
    d.K = K;
    d.hu = hu;
    d.hv = hv;
    d.Gxd = J * hu;
    d.Gxc = J * (v / J);
    d.Gyd = J * hv;
    d.Gyc = J * (-u / J);
    return d;
}

template <typename T>
__device__ __forceinline__ long long pidx(const DevGeo<T> &g, int p, int i, int j) {
    return ((long long)p * g.n + j) * g.pitch + i;
}

// Metric terms of Ah point (i,j) from tan(alpha_i), tan(beta_j), with the operation order of
// the host set-up (ecs_metric_mod.f90:413-463); FP64 only.
struct Metric {
    double J, Qi11, Qi12, Qi22;
};
__device__ __forceinline__ Metric metric_otf(const double *tanA, int i, int j) {
    const double ta = tanA[i], tb = tanA[j];
    const double sg = sqrt(1.0 + ta * ta + tb * tb);
    Metric m;
    m.J = (1.0 + ta * ta) * (1.0 + tb * tb) / (sg * sg * sg);
    m.Qi11 = sg * sg / (1.0 + ta * ta);
    m.Qi12 = sg * sg * ta * tb / ((1 + ta * ta) * (1 + tb * tb));
    m.Qi22 = sg * sg / (1.0 + tb * tb);
    return m;
}

// Element at a byte offset from a uniform base: the offset stays a 32-bit vector register beside a
// scalar base (a panel of the largest grid is 0.54 GB).
template <typename T>
__device__ __forceinline__ T &at_byte(T *base, unsigned off) {
    return *reinterpret_cast<T *>(reinterpret_cast<std::conditional_t<std::is_const_v<T>, const char, char> *>(base) + off);
}

// One panel of the inputs of a stage: state, orography and metric, and the byte offset of a point
template <typename T>
struct PanelIn {
    const T *h, *u, *v, *hs, *J, *q11, *q12, *q22;
    const T *kh, *ku, *kv;   // the stage's input is (h, u, v) + ck (kh, ku, kv) where mode_slope
    T ck;
};
template <typename T>
__device__ __forceinline__ PanelIn<T> panel_in(const DevGeo<T> &g, const StageArgs<T> &a, int p) {
    const long long o = (long long)p * g.n * g.pitch, m = (long long)p * g.mps;
    return {a.y + o, a.y + g.fs + o, a.y + 2 * g.fs + o, a.hs ? a.hs + o : nullptr, g.J + m, g.Qi11 + m, g.Qi12 + m,
            g.Qi22 + m, a.kin + o, a.kin + g.fs + o, a.kin + 2 * g.fs + o, a.ck};
}
template <typename T>
__device__ __forceinline__ unsigned point_off(const DevGeo<T> &g, int i, int j) {
    return (__umul24((unsigned)j, (unsigned)g.pitch) + (unsigned)i) * (unsigned)sizeof(T);
}

// Raw inputs of one point (state, metric, orography) and the derived stencil inputs formed
// from them; split so that the loads of several points can be issued before any is used.
template <typename T>
struct RawPoint {
    T h, u, v, J, q11, q12, q22, hs;
    T kh, ku, kv;
};

template <int MODE, bool OTF, typename T>
__device__ __forceinline__ RawPoint<T> load_point(const DevGeo<T> &g, const PanelIn<T> &in, int i, int j) {
    const unsigned o = point_off(g, i, j);
    RawPoint<T> r;
    r.h = at_byte(in.h, o);
    r.u = at_byte(in.u, o);
    r.v = at_byte(in.v, o);
    if constexpr (mode_slope(MODE)) {
        r.kh = at_byte(in.kh, o);
        r.ku = at_byte(in.ku, o);
        r.kv = at_byte(in.kv, o);
    }
    if constexpr (OTF) {
        const Metric m = metric_otf(g.tanA, i, j);
        r.J = (T)m.J; r.q11 = (T)m.Qi11; r.q12 = (T)m.Qi12; r.q22 = (T)m.Qi22;
    } else {
        r.J = at_byte(in.J, o); r.q11 = at_byte(in.q11, o); r.q12 = at_byte(in.q12, o); r.q22 = at_byte(in.q22, o);
    }
    r.hs = in.hs ? at_byte(in.hs, o) : T(0);
    return r;
}

// r's h, u, v become the stage's input
template <int MODE, typename T>
__device__ __forceinline__ Derived<T> derived_of(const DevGeo<T> &g, RawPoint<T> &r, T ck) {
    if constexpr (mode_slope(MODE)) {
        r.h = r.h + ck * r.kh;
        r.u = r.u + ck * r.ku;
        r.v = r.v + ck * r.kv;
    }
    return make_derived<T>(r.h, r.u, r.v, r.J, r.q11, r.q12, r.q22, r.hs, g.grav);
}

// ----------------------------------------------------------------------------------------
// SBP rows (sbp_operator_mod.f90:187-223).  `get(a)` returns the input at 0-based index a
// along the line; t is the 0-based output index, n the line length.
template <int ORD, int R, typename T, typename G>
__device__ __forceinline__ T sbp_left_row(const G &get) {
    using S = Sbp<ORD>;
    T s = T(S::Ql[R][0]) * get(0);
#pragma unroll
    for (int m = 1; m < S::last[R]; ++m) s = s + T(S::Ql[R][m]) * get(m);
    return s;
}
// right-boundary row ir (0-based): the left row RR = NE-1-ir reflected, sign flipped
template <int ORD, int IR, typename T, typename G>
__device__ __forceinline__ T sbp_right_row(int n, const G &get) {
    using S = Sbp<ORD>;
    constexpr int RR = S::NE - 1 - IR;
    constexpr int LAST = S::last[RR];
    const int base = n - LAST;
    T s = T(-1.0 * S::Ql[RR][LAST - 1]) * get(base);
#pragma unroll
    for (int c = 1; c < LAST; ++c) s = s + T(-1.0 * S::Ql[RR][LAST - 1 - c]) * get(base + c);
    return s;
}

template <int ORD, typename T, typename G, int... Is>
__device__ __forceinline__ T sbp_left_dispatch(int t, const G &get, std::integer_sequence<int, Is...>) {
    T r = T(0);
    ((t == Is ? (void)(r = sbp_left_row<ORD, Is, T>(get)) : (void)0), ...);
    return r;
}
template <int ORD, typename T, typename G, int... Is>
__device__ __forceinline__ T sbp_right_dispatch(int ir, int n, const G &get, std::integer_sequence<int, Is...>) {
    T r = T(0);
    ((ir == Is ? (void)(r = sbp_right_row<ORD, Is, T>(n, get)) : (void)0), ...);
    return r;
}

// interior row of the SBP first derivative at t (NE <= t < n - NE)
template <int ORD, typename T, typename G>
__device__ __forceinline__ T sbp_row_in(int t, const G &get) {
    using S = Sbp<ORD>;
    T s = T(S::Qin[0]) * get(t + S::INSHIFT);
#pragma unroll
    for (int k = 1; k < S::WIN; ++k) s = s + T(S::Qin[k]) * get(t + S::INSHIFT + k);
    return s;
}

template <int ORD, typename T, typename G>
__device__ __forceinline__ T sbp_row(int t, int n, const G &get) {
    using S = Sbp<ORD>;
    if (t >= S::NE && t < n - S::NE) return sbp_row_in<ORD, T>(t, get);
    if (t < S::NE) return sbp_left_dispatch<ORD, T>(t, get, std::make_integer_sequence<int, S::NE>{});
    return sbp_right_dispatch<ORD, T>(t - (n - S::NE), n, get, std::make_integer_sequence<int, S::NE>{});
}

// The rows of the first derivative as a table: classes 0 .. NE-1 the left closure rows, NE the
// interior row, NE+1 .. 2 NE the right closure rows.  Kernels whose points mix the classes read the
// weights from an LDS copy: one code path for every point of a wave, where the rows written out
// with constant weights (sbp_row) take a branch and its code per closure row.
template <int ORD>
struct RowWeights {
    using S = Sbp<ORD>;
    static constexpr int NC = 2 * S::NE + 1, NW = S::NW > S::WIN ? S::NW : S::WIN, SIZE = NC * NW;
    double w[SIZE];
    constexpr RowWeights() : w() {
        for (int r = 0; r < S::NE; ++r)
            for (int m = 0; m < S::last[r]; ++m) {
                w[r * NW + m] = S::Ql[r][m];
                w[(2 * S::NE - r) * NW + m] = -1.0 * S::Ql[r][S::last[r] - 1 - m];
            }
        for (int m = 0; m < S::WIN; ++m) w[S::NE * NW + m] = S::Qin[m];
    }
    static constexpr unsigned packed_last() {
        unsigned v = 0;
        for (int r = 0; r < S::NE; ++r) v |= (unsigned)S::last[r] << (4 * r);
        return v;
    }
};
template <int ORD>
__device__ const RowWeights<ORD> row_weights = RowWeights<ORD>();

// The row of output index t on a line of n points: first input index, number of inputs, class
struct RowAt {
    int base, cnt, cls;
};
template <int ORD>
__device__ __forceinline__ RowAt row_at(int t, int n) {
    using S = Sbp<ORD>;
    constexpr unsigned LASTS = RowWeights<ORD>::packed_last();
    if (t < S::NE) return {0, (int)((LASTS >> (4 * t)) & 15u), t};
    if (t < n - S::NE) return {t + S::INSHIFT, S::WIN, S::NE};
    const int c = (int)((LASTS >> (4 * (n - 1 - t))) & 15u);
    return {n - c, c, 2 * S::NE - (n - 1 - t)};
}
// the row applied to three fields, f(m, a, b, c) giving their inputs at index base + m (reading all
// inputs at once and selecting the sum, without the branch per input, takes 25 VGPRs more: the same
// time on small panels and 2-25 % more on C384)
template <int ORD, typename T, typename F>
__device__ __forceinline__ void row_apply3(const T *__restrict__ tab, const RowAt &r, const F &f, T &a, T &b, T &c) {
    constexpr int NW = RowWeights<ORD>::NW;
    const T *w = tab + r.cls * NW;
    T x, y, z;
    f(0, x, y, z);
    a = w[0] * x;
    b = w[0] * y;
    c = w[0] * z;
#pragma unroll
    for (int m = 1; m < NW; ++m)
        if (m < r.cnt) {
            f(m, x, y, z);
            a = a + w[m] * x;
            b = b + w[m] * y;
            c = c + w[m] * z;
        }
}

// slot of a panel-edge point in a panel's compact edge buffer (4 (n-1) slots)
__device__ __forceinline__ int edge_slot(int n, int i, int j) {
    if (j == 0) return i;
    if (j == n - 1) return n + i;
    if (i == 0) return 2 * n + j - 1;
    return 3 * n + j - 3;
}

// Vector halo convention: neighbour components (a,b) -> local (u,v)
template <typename T>
__device__ __forceinline__ void map_vec(int code, T a, T b, T &u, T &v) {
    const T x = (code & 1) ? b : a;
    const T z = (code & 1) ? a : b;
    u = (code & 2) ? -x : x;
    v = (code & 4) ? -z : z;
}

// XCD-aware mapping: consecutive block ids go round-robin over the 8 XCDs; give each XCD a
// contiguous range of tiles so that tiles sharing halo rows share an L2.
__device__ __forceinline__ int xcd_tile(int bid, int nblocks) {
    const int q = nblocks / 8, r = nblocks % 8;
    const int xcd = bid % 8, local = bid / 8;
    return xcd < r ? xcd * (q + 1) + local : r * (q + 1) + (xcd - r) * q + local;
}

// Order of the tiles of a cube (ntx x nty per panel) whose launch treats tiles with closure rows (the ring) apart
// from the inner ones, columns bx0..bx1-1 of strips by0..by1-1.  A ring tile takes several times an inner
// one; in band order the first and the last XCD would hold a strip of nothing else, and the last one start
// it last.  So the ring goes first, dealt evenly to the XCDs, then the inner tiles, an even share of bands each.
// Within both parts: row strips outermost, then panels, then columns; an XCD's contiguous range is a band of
// all six panels, which read the same metric there.  Up to `slots` tiles, where nearly all blocks are resident
// at once and little waits for a ring tile, all go as ring.  Us alone on the chip, band order / ring first: C-grid
// step C192 112 / 97, C384 243 / 189; hyperdiffusion step C256 sbp42 68 / 48, C384 100 / 77, sbp63 156 / 112;
// transposed RHS with its curl C256 sbp42 27.8 / 23.3, C384 41.9 / 36.8.  Below the lines: C-grid step C64
// 74.9 / 77.3, transposed RHS C192 19.8 / 20.5.  The RK stage kernels stay in band order: their large tiles are a
// third ring, and a C384 step with three contexts at work went from 80 to 81 us (C768 FP32 alone 166 to 155).
struct TileOrder {
    int ntx, nty, bx0, bx1, by0, by1, ring, inner;
    SWM_HD int blocks() const { return ring + inner; }
};
inline TileOrder tile_order(int slots, int ntx, int nty, int bx0, int bx1, int by0, int by1) {
    TileOrder o{ntx, nty, bx0, bx1, by0, by1, 0, 0};
    if (6 * ntx * nty <= slots || bx1 <= bx0 || by1 <= by0) o.bx0 = o.bx1 = o.by0 = o.by1 = 0;
    o.inner = 6 * (o.bx1 - o.bx0) * (o.by1 - o.by0);
    o.ring = 6 * ntx * nty - o.inner;
    return o;
}
// the order for tiles of tx x ty points covering the points first .. first + len - 1 of a panel line of n
// points, inner where all their points lie in margin .. n - 1 - margin
inline TileOrder point_tile_order(int slots, int n, int first, int len, int margin, int tx, int ty) {
    auto lo = [&](int t) { return (margin - first + t - 1) / t; };
    auto hi = [&](int t) { return n - margin - first > 0 ? (n - margin - first) / t : 0; };
    return tile_order(slots, (len + tx - 1) / tx, (len + ty - 1) / ty, lo(tx), hi(tx), lo(ty), hi(ty));
}
struct TilePos {
    int p, cx, cy;
};
// Selects only: with branches here the kernel's other arguments are loaded after them, a second trip to
// memory (0.6 us a launch).
__device__ __forceinline__ TilePos tile_pos(const TileOrder &o, int b) {
    const bool in = b >= o.ring;
    const unsigned nb = in ? o.inner : o.ring, lb = in ? b - o.ring : b;
    // xcd_tile(lb, nb); the inner tiles' shares rotate over the XCDs by ring
    const unsigned q8 = nb / 8, r8 = nb % 8, xcd = lb % 8, extra = xcd < r8 ? xcd : r8;
    unsigned q = xcd * q8 + extra + lb / 8;
    const unsigned wi = o.bx1 - o.bx0, full = 6u * o.ntx * (o.nty - (o.by1 - o.by0));
    const bool sides = !in && q >= full;   // beside the inner tiles of a strip, not a strip without any
    q = sides ? q - full : q;
    const unsigned w = in ? wi : sides ? o.ntx - wi : o.ntx;
    const unsigned s = q / (6 * w), rem = q - s * 6 * w, p = rem / w;
    int cx = rem - p * w, cy = s;
    cx = in || (sides && cx >= o.bx0) ? cx + (in ? o.bx0 : (int)wi) : cx;
    cy = in || sides ? cy + o.by0 : cy >= o.by0 ? cy + (o.by1 - o.by0) : cy;
    return {(int)p, cx, cy};
}

}  // namespace swm
