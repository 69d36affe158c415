// C grid (staggering 'C') vector-invariant shallow-water right-hand side and RK4, SBP42 family:
// divergence_c_sbp42, gradient_c_sbp42, curl_c_sbp42, coriolis_Cgrid_sbp42, KE_Cgrid_sbp42,
// co2contra_c_sbp42, massflux_c_sbp42 (the &shallow_water_model_c set, namelist_swm:80-102),
// composed as operator_swm_t%apply (operator_swm_mod.f90:61-113), FP64.
//
// Points per panel: h at cell centres o (N x N), u at x faces (N+1 x N), v at y faces
// (N x N+1), the curl at corners q (N+1 x N+1).  Every field is stored as 6 panels of
// rows x pitch doubles with a halo of H = 4 on each side; point (i, j) of any type (1-based)
// sits at ((p*rows + j-1+H)*pitch + i-1+H).
//
// The staggered operators are one-dimensional SBP stencils applied along x or y inside a
// panel (sbp_operator_mod.f90:152-228); the panels couple only through
//   - the tangential halo of u and v (curl penalties, curl_c_sbp_mod.f90:73-118),
//   - the face halo of the mass fluxes J*hu, J*hv (divergence penalties,
//     sbp_operator_mod.f90:344-413),
//   - the O-point halo of the kinetic-energy potential (gradient, grad_c_sbp42_mod.f90:53-139),
//   - the corner sync of the curl (halo_Ah_scalar_sync_mod.f90:52-93),
// all read on the fly through precomputed neighbour lists by the tiles on the panel edges.
//
// One RHS is two launches over tiles of TX x TY cells.  k_flux forms the fluxes J hu, J hv, the
// kinetic-energy potential and the raw curl of a tile from the state, k_tend the synced curl, the
// Coriolis terms, the divergence, the gradient, the tendencies and the RK4 stage update from those.
// Every intermediate at another point type (the J Qi12-weighted components and the potential's halves
// in k_flux; the curl at x and y points and the Coriolis terms at o points in k_tend) lives in LDS on
// the tile and the halo that the next stencil reads; only the four fields that need the neighbour
// panels' values go through memory between the two.  Eight launches with the intermediates in
// memory move 91 field passes per step more and leave each launch near its latency floor.
//
// Every expression keeps the reference's operation order with no fused multiply-adds
// (-ffp-contract=off), so results match an FP64 CPU evaluation of the same algorithm bit for bit.

#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>

#include "swm_cctx.h"
#include "swm_reduce.h"

namespace swmc {

constexpr int BX = 16, BY = 16;   // blocks of the diagnostics

// ---- staggered SBP42 operators, sbp_operators_collection_mod.f90:110-191 ----
// W42 interpolation interfaces -> centres, optimised weights (W42_staggered_i2c_opt1)
struct W42i2c {
    static constexpr int NW = 6, NE = 4, INSHIFT = -1, DNX = -1;
    static constexpr double SIGN = 1.0;
    static constexpr int last[4] = {4, 4, 5, 6};
    static constexpr double Ql[4][6] = {
        {0.4892964885611128, 0.48123107353632727, 0.0696483872440123, -0.040175949341450676, 0.0, 0.0},
        {-0.07913099957454726, 0.6127279550862234, 0.5119370885511979, -0.045534044062872786, 0.0, 0.0},
        {-0.0869982983587545, 0.1691760860218048, 0.3626427230326682, 0.6151794893042863, -0.06, 0.0},
        {0.018680545032460714, -0.10869571330417979, 0.09884979151099299, 0.4911653767607321, 0.5625, -0.0625}};
    static constexpr double Qin[4] = {-1.0 / 16.0, 9.0 / 16.0, 9.0 / 16.0, -1.0 / 16.0};
};
// W42 interpolation centres -> interfaces (W42_staggered_c2i_opt1)
struct W42c2i {
    static constexpr int NW = 5, NE = 4, INSHIFT = -2, DNX = 1;
    static constexpr double SIGN = 1.0;
    static constexpr int last[4] = {4, 4, 4, 5};
    static constexpr double Ql[4][5] = {
        {1.3630402181345285, -0.17804474904273135, -0.23303115631809243, 0.048035687226327554, 0.0},
        {0.46340770044238916, 0.4765661872892848, 0.15664452409426372, -0.09661841182593758, 0.0},
        {0.07545241951434666, 0.44794495248229815, 0.37775283649236274, 0.09884979151099299, 0.0},
        {-0.04413695843145285, -0.04040344754874627, 0.649837488701711, 0.4980831989686297, -0.06338028169014084}};
    static constexpr double Qin[4] = {-1.0 / 16.0, 9.0 / 16.0, 9.0 / 16.0, -1.0 / 16.0};
};
// staggered first differences, centres -> interfaces (D42_staggered_c2i)
struct D42c2i {
    static constexpr int NW = 5, NE = 4, INSHIFT = -2, DNX = 1;
    static constexpr double SIGN = -1.0;
    static constexpr int last[4] = {3, 2, 4, 5};
    static constexpr double Ql[4][5] = {{-2.0, 3.0, -1.0, 0.0, 0.0},
                                        {-1.0, 1.0, 0.0, 0.0, 0.0},
                                        {1.0 / 24.0, -9.0 / 8.0, 9.0 / 8.0, -1.0 / 24.0, 0.0},
                                        {-1.0 / 71.0, 6.0 / 71.0, -83.0 / 71.0, 81.0 / 71.0, -3.0 / 71.0}};
    static constexpr double Qin[4] = {1.0 / 24.0, -9.0 / 8.0, 9.0 / 8.0, -1.0 / 24.0};
};
// staggered first differences, interfaces -> centres (D42_staggered_i2c)
struct D42i2c {
    static constexpr int NW = 5, NE = 3, INSHIFT = -1, DNX = -1;
    static constexpr double SIGN = -1.0;
    static constexpr int last[3] = {4, 4, 5};
    static constexpr double Ql[3][5] = {{-79.0 / 78.0, 27.0 / 26.0, -1.0 / 26.0, 1.0 / 78.0, 0.0},
                                        {2.0 / 21.0, -9.0 / 7.0, 9.0 / 7.0, -2.0 / 21.0, 0.0},
                                        {1.0 / 75.0, 0.0, -27.0 / 25.0, 83.0 / 75.0, -1.0 / 25.0}};
    static constexpr double Qin[4] = {1.0 / 24.0, -9.0 / 8.0, 9.0 / 8.0, -1.0 / 24.0};
};

// D42 boundary projection and norms (D42_boundary_proj, D42_A_interfaces, D42_A_centers)
constexpr double PROJ[3] = {15.0 / 8.0, -5.0 / 4.0, 3.0 / 8.0};
constexpr double A_IF1 = 7.0 / 18.0;
// add_penalty_center weights: proj_l(k)/Al_out(k) on the left, proj_r(k)/Ar_out(1+k) on the right
// (Ar_out = A_centers reversed = [1, 25/24, 7/8, 13/12], proj_r = proj_l reversed)
constexpr double PEN_L[3] = {(15.0 / 8.0) / (13.0 / 12.0), (-5.0 / 4.0) / (7.0 / 8.0), (3.0 / 8.0) / (25.0 / 24.0)};
constexpr double PEN_R[3] = {(3.0 / 8.0) / (25.0 / 24.0), (-5.0 / 4.0) / (7.0 / 8.0), (15.0 / 8.0) / (13.0 / 12.0)};

// one output row i (1-based) of sbp_apply along a line with values f(k), k = 1..nsrc: left rows
// sum(Ql(1:last,i) f(1:last)), inner rows sum(Qin f(i+inshift:...)), right rows the left block
// reflected (sign SIGN), each accumulated left to right from the first product
template <class O, class F>
__device__ __forceinline__ double sopf(int i, int nsrc, F &&f) {
    const int ntarg = nsrc + O::DNX;
    double r;
    if (i <= O::NE) {
        const int L = O::last[i - 1];
        r = O::Ql[i - 1][0] * f(1);
#pragma unroll
        for (int m = 2; m <= O::NW; ++m)
            if (m <= L) r = r + O::Ql[i - 1][m - 1] * f(m);
    } else if (i <= ntarg - O::NE) {
        const int b = i + O::INSHIFT;
        r = O::Qin[0] * f(b);
        r = r + O::Qin[1] * f(b + 1);
        r = r + O::Qin[2] * f(b + 2);
        r = r + O::Qin[3] * f(b + 3);
    } else {
        const int l = ntarg - i + 1;  // mirrored left row
        const int L = O::last[l - 1];
        const int b = nsrc + 1 - L;
        r = (O::SIGN * O::Ql[l - 1][L - 1]) * f(b);
#pragma unroll
        for (int t = 1; t < O::NW; ++t)
            if (t < L) r = r + (O::SIGN * O::Ql[l - 1][L - 1 - t]) * f(b + t);
    }
    return r;
}

// the same on a strided array line, f(k) = f0[k*s]
template <class O>
__device__ __forceinline__ double sop(int i, int nsrc, const double *__restrict__ f0, long long s) {
    return sopf<O>(i, nsrc, [&](int k) { return f0[(long long)k * s]; });
}

// ---- the same rows from tables ----
// Classes 0 .. NE-1 the left closure rows, NE the interior row, NE+1 .. 2 NE the right closure rows, NW
// weights each; a tile that holds closure rows reads them from LDS, one code path for all its points.
template <class O>
struct Rows {
    static constexpr int NW = O::NW, NC = 2 * O::NE + 1, SIZE = NC * NW;
    static constexpr void fill(double *w) {
        for (int c = 0; c < SIZE; ++c) w[c] = 0.0;
        for (int r = 0; r < O::NE; ++r)
            for (int m = 0; m < O::last[r]; ++m) {
                w[r * NW + m] = O::Ql[r][m];
                w[(2 * O::NE - r) * NW + m] = O::SIGN * O::Ql[r][O::last[r] - 1 - m];
            }
        for (int m = 0; m < 4; ++m) w[O::NE * NW + m] = O::Qin[m];
    }
    static constexpr unsigned packed_last() {
        unsigned v = 0;
        for (int r = 0; r < O::NE; ++r) v |= (unsigned)O::last[r] << (4 * r);
        return v;
    }
    static constexpr int min_last() {
        int m = 4;
        for (int r = 0; r < O::NE; ++r) m = O::last[r] < m ? O::last[r] : m;
        return m;
    }
    static constexpr int MINLAST = min_last();
};
// the tables of the four operators one after the other
constexpr int ROW_I2C = 0, ROW_C2I = ROW_I2C + Rows<W42i2c>::SIZE, ROW_DC2I = ROW_C2I + Rows<W42c2i>::SIZE,
              ROW_DI2C = ROW_DC2I + Rows<D42c2i>::SIZE, ROW_SIZE = ROW_DI2C + Rows<D42i2c>::SIZE;
template <class O> constexpr int row_start();
template <> constexpr int row_start<W42i2c>() { return ROW_I2C; }
template <> constexpr int row_start<W42c2i>() { return ROW_C2I; }
template <> constexpr int row_start<D42c2i>() { return ROW_DC2I; }
template <> constexpr int row_start<D42i2c>() { return ROW_DI2C; }
struct RowTab {
    double w[ROW_SIZE];
    constexpr RowTab() : w() {
        Rows<W42i2c>::fill(w + ROW_I2C);
        Rows<W42c2i>::fill(w + ROW_C2I);
        Rows<D42c2i>::fill(w + ROW_DC2I);
        Rows<D42i2c>::fill(w + ROW_DI2C);
    }
};
__device__ const RowTab row_tab = RowTab();

// output row i (1-based) of operator O on a line of nsrc inputs f(k): the interior row with constant
// weights (INNER at compile time, or `inner` for a tile whose rows along this line all are), or any row
// from the table
template <class O, bool INNER, class F>
__device__ __forceinline__ double trow(const double *tab, bool inner, int i, int nsrc, const F &f) {
    if (INNER || inner) {
        const int b = i + O::INSHIFT;
        double r = O::Qin[0] * f(b);
        r = r + O::Qin[1] * f(b + 1);
        r = r + O::Qin[2] * f(b + 2);
        return r + O::Qin[3] * f(b + 3);
    } else {
        constexpr unsigned LASTS = Rows<O>::packed_last();
        const int ntarg = nsrc + O::DNX;
        int b = i + O::INSHIFT, cnt = 4, cls = O::NE;
        if (i <= O::NE) {
            b = 1;
            cnt = (int)((LASTS >> (4 * (i - 1))) & 15u);
            cls = i - 1;
        } else if (i > ntarg - O::NE) {
            cnt = (int)((LASTS >> (4 * (ntarg - i))) & 15u);
            b = nsrc + 1 - cnt;
            cls = 2 * O::NE - (ntarg - i);
        }
        const double *w = tab + row_start<O>() + cls * O::NW;
        // all inputs are read at once (the last one again beyond the row's end) and the sum stops at cnt: a
        // branch per input would wait for LDS input by input
        double x[O::NW];
#pragma unroll
        for (int m = 0; m < O::NW; ++m) x[m] = f(b + (m < Rows<O>::MINLAST ? m : min(m, cnt - 1)));
        double r = w[0] * x[0];
#pragma unroll
        for (int m = 1; m < O::NW; ++m) {
            const double z = r + w[m] * x[m];
            r = m < Rows<O>::MINLAST || m < cnt ? z : r;
        }
        return r;
    }
}

// range lo .. hi of points along a line, and the inputs that the rows of a range read (closure rows:
// at most 6 (i2c) / 5 (c2i) points from the end)
struct Rng {
    int lo, hi;
};
template <class O>
__device__ __forceinline__ Rng rng_in(const Rng &r, int nsrc) {
    if (r.lo > r.hi) return {1 << 30, -(1 << 30)};
    const int ntarg = nsrc + O::DNX;
    int lo = r.lo + O::INSHIFT, hi = r.hi + O::INSHIFT + 3;
    if (r.lo <= O::NE) {
        lo = 1;
        hi = max(hi, O::NW);
    }
    if (r.hi > ntarg - O::NE) {
        hi = nsrc;
        lo = min(lo, nsrc + 1 - O::NW);
    }
    return {max(lo, 1), min(hi, nsrc)};
}
__device__ __forceinline__ Rng hull(const Rng &a, const Rng &b) { return {min(a.lo, b.lo), max(a.hi, b.hi)}; }

// metric terms J, Qi at the four point types depend on (alpha, beta) only: one panel plane each,
// read for every panel at the point's offset within its panel (mid); f differs per panel.
// Cube-edge neighbour lists (offsets in the stored layout, signs +-1), indexed by panel p, edge
// e (0: i = 1 side, 1: i = nx side, 2: j = 1 side, 3: j = ny side), depth d and position k:
//   vsrc/vsg  the tangential vector component (v beyond x edges, u beyond y edges), offsets from
//             the u field (+fs for v), [((p*4+e)*3 + d-1)*(N+1) + k-1]
//   fsrc/fsg  the neighbour's copy of a shared face (normal component), from the first field of
//             the pair, [(p*4+e)*N + k-1]
//   osrc      O points, [((p*4+e)*3 + d-1)*N + k-1]
//   qnb       q points on an edge: the neighbour's copy, [(p*4+e)*(N+1) + k-1]
struct CGeo {
    const double *Jo, *Jx, *Jy, *Jq, *Qi12o, *Qi11x, *Qi22y, *JQo, *fo;  // JQo = Jo Qi12o
    const double *hs;  // orography at o points, or NULL
    const long long *vsrc, *fsrc, *osrc, *qnb;
    const signed char *vsg, *fsg;
    int N, pitch;
    int nbx, nby, ntiles, per;  // tiles per row, row strips per panel, tiles, tiles per XCD
    long long plane, fs;
    double hx, scale, grav, dx1;
};

__device__ __forceinline__ long long cid(const CGeo &g, int p, int i, int j) {
    return (long long)p * g.plane + (long long)(j - 1 + H) * g.pitch + (i - 1 + H);
}

// tangential vector component beyond edge e at depth d, position k (pair = u field)
__device__ __forceinline__ double vhalo(const CGeo &g, const double *pair, int p, int e, int d, int k) {
    const long long x = (((long long)p * 4 + e) * 3 + (d - 1)) * (g.N + 1) + (k - 1);
    const double val = pair[g.vsrc[x]];
    return g.vsg[x] < 0 ? -val : val;
}
// the neighbour's copy of the shared face beyond edge e at position k (pair = first field)
__device__ __forceinline__ double fhalo(const CGeo &g, const double *pair, int p, int e, int k) {
    const long long x = ((long long)p * 4 + e) * g.N + (k - 1);
    const double val = pair[g.fsrc[x]];
    return g.fsg[x] < 0 ? -val : val;
}
__device__ __forceinline__ double ohalo(const CGeo &g, const double *f, int p, int e, int d, int k) {
    return f[g.osrc[(((long long)p * 4 + e) * 3 + (d - 1)) * g.N + (k - 1)]];
}

// RK4 stage handling of the tendencies k (rk4_mod.f90:20-42; stage inputs as stvec_swm_t%assign forms
// them): RK_RHS writes k; RK_S1 the next stage input 1.0*v0 + b*k and acc = v0 + c*k; RK_S23 the next
// stage input and acc = acc + c*k; RK_S4 the new state acc + c*k (the reference's sum
// v0 + c2 k0 + c3 k1 + c3 k2 + c2 k3 added up from the left as the stages produce its terms).
enum { RK_RHS = 0, RK_S1 = 1, RK_S23 = 2, RK_S4 = 3 };
struct RkArgs {
    double *out;        // k (RK_RHS), the next stage input, or the new state (RK_S4)
    const double *v0;   // stage-1 state (RK_S1, RK_S23)
    double *acc;
    double b, c;
};
struct RkPre {
    double v0, acc;
};
template <int RKM>
__device__ __forceinline__ RkPre rk_pre(const RkArgs &r, long long base, unsigned off) {
    RkPre q{0.0, 0.0};
    if (RKM == RK_S1 || RKM == RK_S23) q.v0 = swm::at_byte(r.v0 + base, off);
    if (RKM == RK_S23 || RKM == RK_S4) q.acc = swm::at_byte((const double *)r.acc + base, off);
    return q;
}
template <int RKM>
__device__ __forceinline__ void rk_out(const RkArgs &r, long long base, unsigned off, const RkPre &q, double k) {
    if (RKM == RK_RHS) swm::at_byte(r.out + base, off) = k;
    if (RKM == RK_S1 || RKM == RK_S23) {
        swm::at_byte(r.out + base, off) = 1.0 * q.v0 + r.b * k;
        swm::at_byte(r.acc + base, off) = (RKM == RK_S1 ? q.v0 : q.acc) + r.c * k;
    }
    if (RKM == RK_S4) swm::at_byte(r.out + base, off) = q.acc + r.c * k;
}

// Block -> tile mapping: tiles of BX x BY points in the order (column strip fastest, row strip,
// panel); the hardware hands consecutive block indices to the 8 XCDs in turn, so block b takes
// tile (b % 8) * per + b / 8 and every XCD walks a contiguous band of row strips, keeping the
// rows its stencils share in its own L2
#define C_POINT                                                        \
    const int tile_ = (int)(blockIdx.x & 7) * g.per + (int)(blockIdx.x >> 3); \
    if (tile_ >= g.ntiles) return;                                     \
    const int tx_ = tile_ % g.nbx, ty_ = (tile_ / g.nbx) % g.nby;       \
    const int i = tx_ * BX + threadIdx.x + 1;                          \
    const int j = ty_ * BY + threadIdx.y + 1;                          \
    const int p = tile_ / (g.nbx * g.nby);

// ---- tiles ----
// extents of a tile's LDS boxes beyond its TX (TY) cells: faces that the cells' interpolations read (F),
// o points that those faces read (O), o points that the own faces read (C), faces that the C points
// read (Q).  Tiles with closure rows need a little more than tiles of interior rows; the widest over
// every N and tile position (closure rows of the last points reach back over a narrow last tile).
template <bool INNER> constexpr int EXT_F = INNER ? 3 : 5;
template <bool INNER> constexpr int EXT_O = INNER ? 6 : 7;
template <bool INNER> constexpr int EXT_C = INNER ? 3 : 4;
template <bool INNER> constexpr int EXT_Q = INNER ? 6 : 8;

// a tile of panel p: cells x0..x1 x y0..y1, own faces (and q points) up to fx1, fy1: the last tile of a
// line holds the face N+1 too
struct CTile {
    int p, x0, y0, x1, y1, fx1, fy1;
};
// gradient_c_sbp42 along one line at face i (grad_c_sbp42_mod.f90:61-139) of the values F(k): the rows of
// D42c2i, the right closure rows summed from the edge inwards, and on the panel edges the interface
// penalty with the neighbour's values nb[depth]
template <bool INNER, class F>
__device__ __forceinline__ double grad_row(const double *tab, bool inner, int i, int N, double dx1, const F &Fv,
                                           const double (&nb)[3]) {
    constexpr double din[4] = {1.0 / 24.0, -9.0 / 8.0, 9.0 / 8.0, -1.0 / 24.0};
    if (INNER || inner) {
        double r = Fv(i - 2) * din[0];
        r = r + Fv(i - 1) * din[1];
        r = r + Fv(i) * din[2];
        r = r + Fv(i + 1) * din[3];
        return r * dx1;
    } else {
        constexpr unsigned LASTS = Rows<D42c2i>::packed_last();
        const int n = N + 1;
        const bool right = i > n - 4;
        int b = i - 2, s = 1, cnt = 4, cls = 4;
        if (i <= 4) { b = 1; cls = i - 1; }
        else if (right) { b = n - 1; s = -1; cls = n - i; }
        if (cls < 4) cnt = (int)((LASTS >> (4 * cls)) & 15u);
        const double *w = tab + ROW_DC2I + cls * D42c2i::NW;
        double x[D42c2i::NW];
#pragma unroll
        for (int m = 0; m < D42c2i::NW; ++m) x[m] = Fv(b + s * (m < 2 ? m : min(m, cnt - 1)));
        double r = w[0] * x[0];
#pragma unroll
        for (int m = 1; m < D42c2i::NW; ++m) {
            const double z = r + w[m] * x[m];
            r = m < 2 || m < cnt ? z : r;
        }
        r = (s < 0 ? -r : r) * dx1;
        if (i == 1 || i == n) {
            double dh = 0.0;
#pragma unroll
            for (int m = 0; m < 3; ++m) {
                const double own = Fv(i == 1 ? 1 + m : N - m);
                const double x = PROJ[m] * (i == 1 ? own - nb[m] : nb[m] - own);
                dh = m ? dh + x : x;
            }
            r = r + 0.5 * (dh * dx1) / A_IF1;
        }
        return r;
    }
}

// the synced curl (halo_Ah_scalar_sync_mod.f90:52-93) of the q point (i, j): on a cube edge the mean of
// the two panels' raw values, at a cube corner of the three
__device__ __forceinline__ double curl_at(const CGeo &g, const double *__restrict__ W, int p, int i, int j) {
    const int n = g.N + 1;
    const double w = W[cid(g, p, i, j)];
    const bool ex = i == 1 || i == n, ey = j == 1 || j == n;
    if (!ex && !ey) return w;
    const double a = ex ? W[g.qnb[((long long)p * 4 + (i == 1 ? 0 : 1)) * n + j - 1]] : 0.0;
    const double b = ey ? W[g.qnb[((long long)p * 4 + (j == 1 ? 2 : 3)) * n + i - 1]] : 0.0;
    if (ex && ey) return (w + a + b) / 3.0;
    return 0.5 * (w + (ex ? a : b));
}

// One tile configuration: TX x TY cells, NT threads
template <int TX, int TY, int NT>
struct CTiles {
static constexpr int X = TX, Y = TY, THREADS = NT, SLOTS = 512;

// every point (column c, row r, pass k) of a W x R box dealt to the NT threads, the first to thread FROM
template <int W, int R, int FROM = 0, class F>
static __device__ __forceinline__ void each(int tid, const F &f) {
    static_assert((NT & (NT - 1)) == 0, "power of two");
#pragma unroll
    for (int k = 0; k < (W * R + NT - 1) / NT; ++k) {
        const int q = ((tid + NT - FROM) & (NT - 1)) + k * NT;
        if ((k + 1) * NT <= W * R || q < W * R) f(k, q % W, q / W);
    }
}
template <int W, int R> static constexpr int passes() { return (W * R + NT - 1) / NT; }

static __device__ __forceinline__ CTile c_tile(const CGeo &g, const swm::TilePos &at) {
    CTile c;
    c.p = at.p;
    c.x0 = at.cx * TX + 1;
    c.y0 = at.cy * TY + 1;
    c.x1 = min(c.x0 + TX - 1, g.N);
    c.y1 = min(c.y0 + TY - 1, g.N);
    c.fx1 = c.x1 + (c.x1 == g.N);
    c.fy1 = c.y1 + (c.y1 == g.N);
    return c;
}
// inner tiles: full ones all of whose rows are interior ones (7 <= x0, x1 <= N - 5)
static swm::TileOrder order(int N) {
    return swm::tile_order(SLOTS, (N + TX - 1) / TX, (N + TY - 1) / TY, (6 + TX - 1) / TX, (N - 5) / TX, (6 + TY - 1) / TY, (N - 5) / TY);
}
static __device__ __forceinline__ bool c_inner(const CGeo &g, const CTile &c) {
    return c.x0 >= 7 && c.y0 >= 7 && c.x1 <= g.N - 5 && c.y1 <= g.N - 5 && c.x1 - c.x0 == TX - 1 && c.y1 - c.y0 == TY - 1;
}
static __device__ __forceinline__ unsigned c_off(const CGeo &g, int i, int j) {
    return (__umul24((unsigned)(j - 1 + H), (unsigned)g.pitch) + (unsigned)(i - 1 + H)) * 8u;
}
static __device__ __forceinline__ void load_row_tab(double *tab, int tid) {
    for (int c = tid; c < ROW_SIZE; c += NT) tab[c] = row_tab.w[c];
}

template <bool INNER>
struct FluxSmem {
    static constexpr int F = EXT_F<INNER>, O = EXT_O<INNER>, C = EXT_C<INNER>;
    double u[TY + O][TX + F], v[TY + F][TX + O], h[TY + C][TX + C];
    double A[TY][TX + O], B[TY + O][TX];         // J Qi12-weighted components at o points
    double ku[TY][TX + F], kv[TY + F][TX];       // halves of the potential at x and y points
};

// co2contra_c_sbp42 (co2contra_Cgrid_mod.f90:361-398), massflux_c_sbp42 (massflux_Cgrid_mod.f90:330-355),
// the J-weighted fluxes G = (J hu, J hv) of the divergence and Coriolis terms (div_c_sbp42_mod.f90:
// 101-130, coriolis_Cgrid_mod.f90:69-84), KE_Cgrid (KE_Cgrid_mod.f90:41-75) with the update of
// operator_swm_mod.f90:85, and curl_c_sbp42 before the corner sync (curl_c_sbp_mod.f90:73-118)
template <bool INNER>
static __device__ __forceinline__ void flux_tile(const CGeo &g, const double *__restrict__ y, double *__restrict__ G,
                                          double *__restrict__ KE, double *__restrict__ W, const CTile &t,
                                          FluxSmem<INNER> &sm, double *tab) {
    constexpr int F = EXT_F<INNER>, O = EXT_O<INNER>, C = EXT_C<INNER>;
    const int N = g.N, tid = threadIdx.x, x0 = t.x0, y0 = t.y0, x1 = t.x1, y1 = t.y1;
    const bool inx = INNER || (x0 >= 7 && x1 <= N - 5), iny = INNER || (y0 >= 7 && y1 <= N - 5);
    Rng FX{x0 - 1, x1 + 2}, FY{y0 - 1, y1 + 2}, OX{x0 - 3, x1 + 3}, OY{y0 - 3, y1 + 3}, CX{x0 - 2, x1 + 1}, CY{y0 - 2, y1 + 1};
    if constexpr (!INNER) {
        const Rng fx{x0, t.fx1}, fy{y0, t.fy1};
        FX = hull(rng_in<W42i2c>({x0, x1}, N + 1), fx);
        FY = hull(rng_in<W42i2c>({y0, y1}, N + 1), fy);
        OX = rng_in<W42c2i>(FX, N);
        OY = rng_in<W42c2i>(FY, N);
        CX = rng_in<W42c2i>(fx, N);
        CY = rng_in<W42c2i>(fy, N);
    }
    const long long pb = (long long)t.p * g.plane;
    const double *h = y + pb, *u = y + g.fs + pb, *v = y + 2 * g.fs + pb;
    auto in = [&](int i, int j, const Rng &X, const Rng &Y) { return INNER || (i <= X.hi && j <= Y.hi); };

    // the state on the boxes and the metric at the points where the later phases use it, all in flight
    // together
    double ru[passes<TX + F, TY + O>()], rv[passes<TX + O, TY + F>()], rh[passes<TX + C, TY + C>()];
    double mA[passes<TX + O, TY>()], mB[passes<TX, TY + O>()];
    double q11[passes<TX + F, TY>()], jx[passes<TX + F, TY>()], q22[passes<TX, TY + F>()], jy[passes<TX, TY + F>()];
    each<TX + F, TY + O>(tid, [&](int k, int c, int r) {
        if (in(FX.lo + c, OY.lo + r, FX, OY)) ru[k] = swm::at_byte(u, c_off(g, FX.lo + c, OY.lo + r));
    });
    each<TX + O, TY + F>(tid, [&](int k, int c, int r) {
        if (in(OX.lo + c, FY.lo + r, OX, FY)) rv[k] = swm::at_byte(v, c_off(g, OX.lo + c, FY.lo + r));
    });
    each<TX + C, TY + C>(tid, [&](int k, int c, int r) {
        if (in(CX.lo + c, CY.lo + r, CX, CY)) rh[k] = swm::at_byte(h, c_off(g, CX.lo + c, CY.lo + r));
    });
    const Rng cx{x0, x1}, cy{y0, y1};
    each<TX + O, TY>(tid, [&](int k, int c, int r) {
        if (in(OX.lo + c, y0 + r, OX, cy)) mA[k] = swm::at_byte(g.JQo, c_off(g, OX.lo + c, y0 + r));
    });
    each<TX, TY + O>(tid, [&](int k, int c, int r) {
        if (in(x0 + c, OY.lo + r, cx, OY)) mB[k] = swm::at_byte(g.JQo, c_off(g, x0 + c, OY.lo + r));
    });
    each<TX + F, TY>(tid, [&](int k, int c, int r) {
        if (in(FX.lo + c, y0 + r, FX, cy)) {
            const unsigned o = c_off(g, FX.lo + c, y0 + r);
            q11[k] = swm::at_byte(g.Qi11x, o);
            jx[k] = swm::at_byte(g.Jx, o);
        }
    });
    each<TX, TY + F>(tid, [&](int k, int c, int r) {
        if (in(x0 + c, FY.lo + r, cx, FY)) {
            const unsigned o = c_off(g, x0 + c, FY.lo + r);
            q22[k] = swm::at_byte(g.Qi22y, o);
            jy[k] = swm::at_byte(g.Jy, o);
        }
    });
    // the neighbour's tangential components beyond the panel edges, for the curl's penalties
    double nx[3], ny[3];
    if constexpr (!INNER) {
        static_assert((TX + 1) * (TY + 1) <= NT, "one q point per thread");
        each<TX + 1, TY + 1, NT - TX * TY>(tid, [&](int, int c, int r) {
            const int i = x0 + c, j = y0 + r;
            if (i > t.fx1 || j > t.fy1) return;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if (i == 1 || i == N + 1) nx[k] = vhalo(g, y + g.fs, t.p, i == 1 ? 0 : 1, k + 1, j);
                if (j == 1 || j == N + 1) ny[k] = vhalo(g, y + g.fs, t.p, j == 1 ? 2 : 3, k + 1, i);
            }
        });
    }
    each<TX + F, TY + O>(tid, [&](int k, int c, int r) {
        if (in(FX.lo + c, OY.lo + r, FX, OY)) sm.u[r][c] = ru[k];
    });
    each<TX + O, TY + F>(tid, [&](int k, int c, int r) {
        if (in(OX.lo + c, FY.lo + r, OX, FY)) sm.v[r][c] = rv[k];
    });
    each<TX + C, TY + C>(tid, [&](int k, int c, int r) {
        if (in(CX.lo + c, CY.lo + r, CX, CY)) sm.h[r][c] = rh[k];
    });
    if constexpr (!INNER) load_row_tab(tab, tid);
    __syncthreads();

    each<TX + O, TY>(tid, [&](int k, int c, int r) {
        const int j = y0 + r;
        if (in(OX.lo + c, j, OX, cy))
            sm.A[r][c] = mA[k] * trow<W42i2c, INNER>(tab, iny, j, N + 1, [&](int q) { return sm.v[q - FY.lo][c]; });
    });
    each<TX, TY + O>(tid, [&](int k, int c, int r) {
        const int i = x0 + c;
        if (in(i, OY.lo + r, cx, OY))
            sm.B[r][c] = mB[k] * trow<W42i2c, INNER>(tab, inx, i, N + 1, [&](int q) { return sm.u[r][q - FX.lo]; });
    });
    __syncthreads();

    each<TX + F, TY>(tid, [&](int k, int c, int r) {
        const int i = FX.lo + c, j = y0 + r;
        if (!in(i, j, FX, cy)) return;
        const double tt = trow<W42c2i, INNER>(tab, inx, i, N, [&](int q) { return sm.A[r][q - OX.lo]; });
        const double uu = sm.u[j - OY.lo][c], ut = q11[k] * uu + tt / jx[k];
        sm.ku[r][c] = jx[k] * (uu * ut) / 2.0;
        if (i >= x0 && i <= t.fx1) {
            const double hh = trow<W42c2i, INNER>(tab, inx, i, N, [&](int q) { return sm.h[j - CY.lo][q - CX.lo]; });
            const double hu = ut * hh;
            swm::at_byte(G + pb, c_off(g, i, j)) = jx[k] * hu;
        }
    });
    each<TX, TY + F>(tid, [&](int k, int c, int r) {
        const int i = x0 + c, j = FY.lo + r;
        if (!in(i, j, cx, FY)) return;
        const double tt = trow<W42c2i, INNER>(tab, iny, j, N, [&](int q) { return sm.B[q - OY.lo][c]; });
        const double vv = sm.v[r][i - OX.lo], vt = q22[k] * vv + tt / jy[k];
        sm.kv[r][c] = jy[k] * (vv * vt) / 2.0;
        if (j >= y0 && j <= t.fy1) {
            const double hh = trow<W42c2i, INNER>(tab, iny, j, N, [&](int q) { return sm.h[q - CY.lo][i - CX.lo]; });
            const double hv = vt * hh;
            swm::at_byte(G + g.fs + pb, c_off(g, i, j)) = jy[k] * hv;
        }
    });
    __syncthreads();

    each<TX, TY>(tid, [&](int, int c, int r) {
        const int i = x0 + c, j = y0 + r;
        if (!in(i, j, cx, cy)) return;
        const unsigned o = c_off(g, i, j);
        const double kuh = trow<W42i2c, INNER>(tab, inx, i, N + 1, [&](int q) { return sm.ku[r][q - FX.lo]; });
        const double kvh = trow<W42i2c, INNER>(tab, iny, j, N + 1, [&](int q) { return sm.kv[q - FY.lo][c]; });
        double ke = (kuh + kvh) / swm::at_byte(g.Jo, o);
        ke = ke + g.grav * sm.h[j - CY.lo][i - CX.lo] + g.grav * (g.hs ? swm::at_byte(g.hs + pb, o) : 0.0);
        swm::at_byte(KE + pb, o) = ke;
    });
    // curl: staggered differences of v along x and u along y with the interface penalties, the
    // neighbour's tangential components read through vsrc
    each<INNER ? TX : TX + 1, INNER ? TY : TY + 1, NT - TX * TY>(tid, [&](int, int c, int r) {
        const int i = x0 + c, j = y0 + r, n = N + 1;
        if (!INNER && (i > t.fx1 || j > t.fy1)) return;
        const unsigned o = c_off(g, i, j);
        auto vx = [&](int q) { return sm.v[j - FY.lo][q - OX.lo]; };
        auto uy = [&](int q) { return sm.u[q - OY.lo][i - FX.lo]; };
        double dvx = trow<D42c2i, INNER>(tab, inx, i, N, vx);
        double duy = trow<D42c2i, INNER>(tab, iny, j, N, uy);
        if constexpr (!INNER) {
            if (i == 1 || i == n) {
                double d = 0.0;
#pragma unroll
                for (int k = 1; k <= 3; ++k) d = d + PROJ[k - 1] * (i == 1 ? vx(k) - nx[k - 1] : nx[k - 1] - vx(n - k));
                dvx = dvx + 0.5 * d / A_IF1;
            }
            if (j == 1 || j == n) {
                double d = 0.0;
#pragma unroll
                for (int k = 1; k <= 3; ++k) d = d + PROJ[k - 1] * (j == 1 ? uy(k) - ny[k - 1] : ny[k - 1] - uy(n - k));
                duy = duy + 0.5 * d / A_IF1;
            }
        }
        swm::at_byte(W + pb, o) = (dvx - duy) / (swm::at_byte(g.Jq, o) * g.hx * g.scale);
    });
}

template <bool INNER>
struct TendSmem {
    static constexpr int F = EXT_F<INNER>, C = EXT_C<INNER>, Q = EXT_Q<INNER>;
    double W[TY + Q][TX + Q], gu[TY + C][TX + F], gv[TY + F][TX + C], ke[TY + C][TX + C];
    double fu[TY + C][TX + Q], fv[TY + Q][TX + C];   // the synced curl at x and y points
    double cu[TY][TX + C], cv[TY + C][TX];           // Coriolis terms at o points
};

// interpolator_w2h of the synced curl (interpolator_w2h_mod.f90:40-68), the vector-invariant Coriolis
// terms (coriolis_Cgrid_mod.f90:86-103) and their interpolation to faces (interpolator_p2uv_mod.f90:
// 90-113), dh = -div(J hu, J hv) with the centre penalties (div_c_sbp42_mod.f90:70-99,
// sbp_operator_mod.f90:344-413), du = -grad_x(KE) + cor_u, dv = -grad_y(KE) + cor_v
// (operator_swm_mod.f90:94-95), and the RK4 stage update
template <int RKM, bool INNER>
static __device__ __forceinline__ void tend_tile(const CGeo &g, const double *__restrict__ h, const double *__restrict__ G,
                                          const double *__restrict__ KE, const double *__restrict__ W,
                                          const RkArgs &rk, const CTile &t, TendSmem<INNER> &sm, double *tab) {
    constexpr int F = EXT_F<INNER>, C = EXT_C<INNER>, Q = EXT_Q<INNER>;
    const int N = g.N, tid = threadIdx.x, x0 = t.x0, y0 = t.y0, x1 = t.x1, y1 = t.y1;
    const bool inx = INNER || (x0 >= 7 && x1 <= N - 5), iny = INNER || (y0 >= 7 && y1 <= N - 5);
    Rng GX{x0 - 1, x1 + 2}, GY{y0 - 1, y1 + 2}, CX{x0 - 2, x1 + 1}, CY{y0 - 2, y1 + 1}, QX{x0 - 3, x1 + 3}, QY{y0 - 3, y1 + 3};
    const Rng cx{x0, x1}, cy{y0, y1};
    if constexpr (!INNER) {
        GX = rng_in<W42i2c>(cx, N + 1);
        GY = rng_in<W42i2c>(cy, N + 1);
        CX = hull(rng_in<W42c2i>({x0, t.fx1}, N), cx);
        CY = hull(rng_in<W42c2i>({y0, t.fy1}, N), cy);
        QX = rng_in<W42i2c>(CX, N + 1);
        QY = rng_in<W42i2c>(CY, N + 1);
    }
    const long long pb = (long long)t.p * g.plane;
    auto in = [&](int i, int j, const Rng &X, const Rng &Y) { return INNER || (i <= X.hi && j <= Y.hi); };

    // the four fields on the boxes, and the own points' stage vectors and the o points' f and h, all in
    // flight together
    double rw[passes<TX + Q, TY + Q>()], ru[passes<TX + F, TY + C>()], rv[passes<TX + C, TY + F>()], re[passes<TX + C, TY + C>()];
    double fa[passes<TX + C, TY>()], ha[passes<TX + C, TY>()], fb[passes<TX, TY + C>()], hb[passes<TX, TY + C>()];
    each<TX + Q, TY + Q>(tid, [&](int k, int c, int r) {
        const int i = QX.lo + c, j = QY.lo + r;
        if (INNER) rw[k] = swm::at_byte(W + pb, c_off(g, i, j));
        else if (in(i, j, QX, QY)) rw[k] = curl_at(g, W, t.p, i, j);
    });
    each<TX + F, TY + C>(tid, [&](int k, int c, int r) {
        if (in(GX.lo + c, CY.lo + r, GX, CY)) ru[k] = swm::at_byte(G + pb, c_off(g, GX.lo + c, CY.lo + r));
    });
    each<TX + C, TY + F>(tid, [&](int k, int c, int r) {
        if (in(CX.lo + c, GY.lo + r, CX, GY)) rv[k] = swm::at_byte(G + g.fs + pb, c_off(g, CX.lo + c, GY.lo + r));
    });
    each<TX + C, TY + C>(tid, [&](int k, int c, int r) {
        if (in(CX.lo + c, CY.lo + r, CX, CY)) re[k] = swm::at_byte(KE + pb, c_off(g, CX.lo + c, CY.lo + r));
    });
    each<TX + C, TY>(tid, [&](int k, int c, int r) {
        if (!in(CX.lo + c, y0 + r, CX, cy)) return;
        const unsigned o = c_off(g, CX.lo + c, y0 + r);
        fa[k] = swm::at_byte(g.fo + pb, o);
        ha[k] = swm::at_byte(h + pb, o);
    });
    each<TX, TY + C>(tid, [&](int k, int c, int r) {
        if (!in(x0 + c, CY.lo + r, cx, CY)) return;
        const unsigned o = c_off(g, x0 + c, CY.lo + r);
        fb[k] = swm::at_byte(g.fo + pb, o);
        hb[k] = swm::at_byte(h + pb, o);
    });
    // the neighbours' values that the penalties of the own points read: copies of the shared faces (nx, ny),
    // the potential beyond the x edges (ex) and the y edges (ey)
    double nx = 0.0, ny = 0.0, ex[3], ey[3];
    if constexpr (!INNER) {
        static_assert((TX + 1) * (TY + 1) <= NT, "one point of each type per thread");
        each<TX, TY>(tid, [&](int, int c, int r) {
            const int i = x0 + c, j = y0 + r;
            if (!in(i, j, cx, cy)) return;
            if (i <= 3 || i >= N - 2) nx = fhalo(g, G, t.p, i <= 3 ? 0 : 1, j);
            if (j <= 3 || j >= N - 2) ny = fhalo(g, G, t.p, j <= 3 ? 2 : 3, i);
        });
        each<TX + 1, TY, NT - TX * TY>(tid, [&](int, int c, int r) {
            const int i = x0 + c, j = y0 + r;
            if ((i == 1 || i == N + 1) && j <= y1)
#pragma unroll
                for (int k = 0; k < 3; ++k) ex[k] = ohalo(g, KE, t.p, i == 1 ? 0 : 1, k + 1, j);
        });
        each<TX, TY + 1>(tid, [&](int, int c, int r) {
            const int i = x0 + c, j = y0 + r;
            if ((j == 1 || j == N + 1) && i <= x1)
#pragma unroll
                for (int k = 0; k < 3; ++k) ey[k] = ohalo(g, KE, t.p, j == 1 ? 2 : 3, k + 1, i);
        });
    }
    each<TX + Q, TY + Q>(tid, [&](int k, int c, int r) {
        if (in(QX.lo + c, QY.lo + r, QX, QY)) sm.W[r][c] = rw[k];
    });
    each<TX + F, TY + C>(tid, [&](int k, int c, int r) {
        if (in(GX.lo + c, CY.lo + r, GX, CY)) sm.gu[r][c] = ru[k];
    });
    each<TX + C, TY + F>(tid, [&](int k, int c, int r) {
        if (in(CX.lo + c, GY.lo + r, CX, GY)) sm.gv[r][c] = rv[k];
    });
    each<TX + C, TY + C>(tid, [&](int k, int c, int r) {
        if (in(CX.lo + c, CY.lo + r, CX, CY)) sm.ke[r][c] = re[k];
    });
    if constexpr (!INNER) load_row_tab(tab, tid);
    __syncthreads();

    each<TX + Q, TY + C>(tid, [&](int, int c, int r) {
        const int j = CY.lo + r;
        if (in(QX.lo + c, j, QX, CY))
            sm.fu[r][c] = trow<W42i2c, INNER>(tab, iny, j, N + 1, [&](int q) { return sm.W[q - QY.lo][c]; });
    });
    each<TX + C, TY + Q>(tid, [&](int, int c, int r) {
        const int i = CX.lo + c;
        if (in(i, QY.lo + r, CX, QY))
            sm.fv[r][c] = trow<W42i2c, INNER>(tab, inx, i, N + 1, [&](int q) { return sm.W[r][q - QX.lo]; });
    });
    __syncthreads();

    // curl_p = (I_x fu + I_y fv)/2 at the o point (i, j)
    auto curl_p = [&](int i, int j) {
        const double fuh = trow<W42i2c, INNER>(tab, inx, i, N + 1, [&](int q) { return sm.fu[j - CY.lo][q - QX.lo]; });
        const double fvh = trow<W42i2c, INNER>(tab, iny, j, N + 1, [&](int q) { return sm.fv[q - QY.lo][i - CX.lo]; });
        return 0.5 * fuh + 0.5 * fvh;
    };
    each<TX + C, TY>(tid, [&](int k, int c, int r) {
        const int i = CX.lo + c, j = y0 + r;
        if (!in(i, j, CX, cy)) return;
        const double gv = trow<W42i2c, INNER>(tab, iny, j, N + 1, [&](int q) { return sm.gv[q - GY.lo][c]; });
        sm.cu[r][c] = (fa[k] + curl_p(i, j)) * gv / ha[k];
    });
    each<TX, TY + C>(tid, [&](int k, int c, int r) {
        const int i = x0 + c, j = CY.lo + r;
        if (!in(i, j, cx, CY)) return;
        const double gu = trow<W42i2c, INNER>(tab, inx, i, N + 1, [&](int q) { return sm.gu[r][q - GX.lo]; });
        sm.cv[r][c] = -(fb[k] + curl_p(i, j)) * gu / hb[k];
    });
    // the stage vectors of the own points, in flight across the barrier (tiles of interior rows: one
    // point of each field per thread)
    RkPre qh{}, qu{}, qv{};
    if constexpr (INNER) {
        const int m = tid & (TX * TY - 1);   // the own point, as the loops below deal them
        const unsigned o = c_off(g, x0 + m % TX, y0 + m / TX);
        if (tid < TX * TY) {
            qh = rk_pre<RKM>(rk, pb, o);
            qv = rk_pre<RKM>(rk, 2 * g.fs + pb, o);
        }
        if (tid >= NT - TX * TY) qu = rk_pre<RKM>(rk, g.fs + pb, o);
    }
    __syncthreads();

    each<TX, TY>(tid, [&](int, int c, int r) {
        const int i = x0 + c, j = y0 + r;
        if (!in(i, j, cx, cy)) return;
        const unsigned o = c_off(g, i, j);
        auto gx = [&](int q) { return sm.gu[j - CY.lo][q - GX.lo]; };
        auto gy = [&](int q) { return sm.gv[q - GY.lo][i - CX.lo]; };
        double dx = trow<D42i2c, INNER>(tab, inx, i, N + 1, gx);
        double dy = trow<D42i2c, INNER>(tab, iny, j, N + 1, gy);
        if constexpr (!INNER) {
            if (i <= 3) dx = dx + 0.5 * PEN_L[i - 1] * (gx(1) - nx);
            if (i >= N - 2) dx = dx + 0.5 * PEN_R[i - N + 2] * (nx - gx(N + 1));
            if (j <= 3) dy = dy + 0.5 * PEN_L[j - 1] * (gy(1) - ny);
            if (j >= N - 2) dy = dy + 0.5 * PEN_R[j - N + 2] * (ny - gy(N + 1));
            qh = rk_pre<RKM>(rk, pb, o);
        }
        const double div = (dx + dy) / (swm::at_byte(g.Jo, o) * g.hx * g.scale);
        rk_out<RKM>(rk, pb, o, qh, -1.0 * div);
    });
    each<INNER ? TX : TX + 1, TY, NT - TX * TY>(tid, [&](int, int c, int r) {
        const int i = x0 + c, j = y0 + r;
        if (!INNER && (i > t.fx1 || j > y1)) return;
        const unsigned o = c_off(g, i, j);
        const double gx = grad_row<INNER>(tab, inx, i, N, g.dx1, [&](int q) { return sm.ke[j - CY.lo][q - CX.lo]; }, ex);
        const double cu = trow<W42c2i, INNER>(tab, inx, i, N, [&](int q) { return sm.cu[r][q - CX.lo]; });
        if constexpr (!INNER) qu = rk_pre<RKM>(rk, g.fs + pb, o);
        rk_out<RKM>(rk, g.fs + pb, o, qu, -1.0 * gx + 1.0 * cu);
    });
    each<TX, INNER ? TY : TY + 1>(tid, [&](int, int c, int r) {
        const int i = x0 + c, j = y0 + r;
        if (!INNER && (i > x1 || j > t.fy1)) return;
        const unsigned o = c_off(g, i, j);
        const double gy = grad_row<INNER>(tab, iny, j, N, g.dx1, [&](int q) { return sm.ke[q - CY.lo][i - CX.lo]; }, ey);
        const double cv = trow<W42c2i, INNER>(tab, iny, j, N, [&](int q) { return sm.cv[q - CY.lo][c]; });
        if constexpr (!INNER) qv = rk_pre<RKM>(rk, 2 * g.fs + pb, o);
        rk_out<RKM>(rk, 2 * g.fs + pb, o, qv, -1.0 * gy + 1.0 * cv);
    });
}

};

// 16 x 8 cells and two threads per cell: the phases of a tile have 1.3 to 3 tasks per cell, a block is a
// chain of load, three LDS phases and stores whose length is what a launch of few tiles takes, and 8 such
// blocks fit a CU.  RK4 step (8 launches), C90 / C384 / C512: 74 / 241 / 365 us in plain band order, 75 / 191 / 306
// with the ring first (TileOrder: 29 and 35 us a launch at C384, 24 and 29 then); in band order 8 x 8 cells
// 75 / 342 / 537, 32 x 4 69 / 273 / 406, 32 x 8 with 512 threads 85 / 306 / 460, with 256 124 / 287 / 383; the
// eight-launch form with its intermediates in memory 140 / 391 us.
using Tiles = CTiles<16, 8, 256>;

__global__ void __launch_bounds__(Tiles::THREADS) k_flux(swm::TileOrder order, CGeo g, const double *__restrict__ y, double *__restrict__ G,
                                                         double *__restrict__ KE, double *__restrict__ W) {
    __shared__ union { Tiles::FluxSmem<true> in; Tiles::FluxSmem<false> any; } sm;
    __shared__ double tab[ROW_SIZE];
    const CTile t = Tiles::c_tile(g, swm::tile_pos(order, blockIdx.x));
    if (Tiles::c_inner(g, t)) Tiles::flux_tile<true>(g, y, G, KE, W, t, sm.in, tab);
    else Tiles::flux_tile<false>(g, y, G, KE, W, t, sm.any, tab);
}

template <int RKM>
__global__ void __launch_bounds__(Tiles::THREADS) k_tend(swm::TileOrder order, CGeo g, const double *__restrict__ h, const double *__restrict__ G,
                                                            const double *__restrict__ KE, const double *__restrict__ W,
                                                            RkArgs r) {
    __shared__ union { Tiles::TendSmem<true> in; Tiles::TendSmem<false> any; } sm;
    __shared__ double tab[ROW_SIZE];
    const CTile t = Tiles::c_tile(g, swm::tile_pos(order, blockIdx.x));
    if (Tiles::c_inner(g, t)) Tiles::tend_tile<RKM, true>(g, h, G, KE, W, r, t, sm.in, tab);
    else Tiles::tend_tile<RKM, false>(g, h, G, KE, W, r, t, sm.any, tab);
}

// ---- get_diagnostics on the C grid (operator_swm_mod.f90:115-155, calc_energy :211-236) ----
// Per-point terms f*J*hx*hy*Ax(i)*Ay(j) of SBP_C42_quadrature (sbp_quadrature_mod.f90:21-40;
// Ax, Ay = A_centers along centre directions, A_interfaces along face directions) summed with
// compensated (Neumaier) additions per block: mass, KE_u, KE_v, PE, then hmin, hmax.
constexpr int CD_NQ = 4;

__global__ void __launch_bounds__(256) k_cdiag_partial(CGeo g, const double *__restrict__ y,
                                                       const double *__restrict__ Acen,
                                                       const double *__restrict__ Aint, double *__restrict__ part) {
    C_POINT
    const int N = g.N;
    const double *h = y, *u = y + g.fs, *v = y + 2 * g.fs;
    double s[CD_NQ] = {0.0, 0.0, 0.0, 0.0}, cc[CD_NQ] = {0.0, 0.0, 0.0, 0.0};
    double hmin = 1e300, hmax = -1e300;
    const double hx = g.hx;
    if (i <= N && j <= N) {
        const long long id = cid(g, p, i, j), mid = id - (long long)p * g.plane;
        const double hh = h[id];
        hmin = hh;
        hmax = hh;
        swm::neu_add(s[0], cc[0], hh * g.Jo[mid] * hx * hx * Acen[i] * Acen[j]);
        const double pe = 1.0 * hh + 1.0 * (g.hs ? g.hs[id] : 0.0);
        const double PE = 0.5 * g.grav * pe * pe;
        swm::neu_add(s[3], cc[3], PE * g.Jo[mid] * hx * hx * Acen[i] * Acen[j]);
    }
    if (i <= N + 1 && j <= N) {  // KE_diag_u = 0.5 * hu * u at x points, hu = massflux(h, ut)
        const long long id = cid(g, p, i, j), mid = id - (long long)p * g.plane;
        const double t = sopf<W42c2i>(i, N, [&](int ip) {
            const long long m = cid(g, 0, ip, j);
            const double dy = sop<W42i2c>(j, N + 1, v + cid(g, p, ip, 0), g.pitch);
            return g.Jo[m] * g.Qi12o[m] * dy;
        });
        const double ut = g.Qi11x[mid] * u[id] + t / g.Jx[mid];
        const double hu = ut * sop<W42c2i>(i, N, h + cid(g, p, 0, j), 1);
        const double ke = 0.5 * hu * u[id];
        swm::neu_add(s[1], cc[1], ke * g.Jx[mid] * hx * hx * Aint[i] * Acen[j]);
    }
    if (i <= N && j <= N + 1) {
        const long long id = cid(g, p, i, j), mid = id - (long long)p * g.plane;
        const double t = sopf<W42c2i>(j, N, [&](int jp) {
            const long long m = cid(g, 0, i, jp);
            const double dx = sop<W42i2c>(i, N + 1, u + cid(g, p, 0, jp), 1);
            return g.Jo[m] * g.Qi12o[m] * dx;
        });
        const double vt = g.Qi22y[mid] * v[id] + t / g.Jy[mid];
        const double hv = vt * sop<W42c2i>(j, N, h + cid(g, p, i, 0), g.pitch);
        const double ke = 0.5 * hv * v[id];
        swm::neu_add(s[2], cc[2], ke * g.Jy[mid] * hx * hx * Acen[i] * Aint[j]);
    }
    __shared__ double sh[256][2 * CD_NQ + 2];
    const int t = threadIdx.y * BX + threadIdx.x;
    for (int q = 0; q < CD_NQ; ++q) {
        sh[t][2 * q] = s[q];
        sh[t][2 * q + 1] = cc[q];
    }
    sh[t][2 * CD_NQ] = hmin;
    sh[t][2 * CD_NQ + 1] = hmax;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) {
            for (int q = 0; q < CD_NQ; ++q) {
                double a = sh[t][2 * q], ac = sh[t][2 * q + 1];
                swm::neu_add(a, ac, sh[t + w][2 * q]);
                ac += sh[t + w][2 * q + 1];
                sh[t][2 * q] = a;
                sh[t][2 * q + 1] = ac;
            }
            sh[t][2 * CD_NQ] = fmin(sh[t][2 * CD_NQ], sh[t + w][2 * CD_NQ]);
            sh[t][2 * CD_NQ + 1] = fmax(sh[t][2 * CD_NQ + 1], sh[t + w][2 * CD_NQ + 1]);
        }
        __syncthreads();
    }
    if (t < 2 * CD_NQ + 2) part[(long long)t * g.ntiles + tile_] = sh[0][t];
}

// the block partials summed by one block: {mass, KE_u, KE_v, PE, hmin, hmax}
__global__ void __launch_bounds__(swm::FINAL_THREADS) k_cdiag_final(const double *__restrict__ part, long long nblocks,
                                                                    double *__restrict__ out) {
    swm::sum_partials<CD_NQ>(part, nblocks, out);
}

#undef C_POINT

}  // namespace swmc

// ------------------------------------------------------------------------------------------------
namespace {

constexpr int CW_G = 0 /* and 1 */, CW_KE = 2, CW_W = 3, CW_ACC = 4, CW_YA = 7, CW_YB = 10, CW_COUNT = 13;

swmc::CGeo make_cgeo(const swm_cctx *c) {
    swmc::CGeo g;
    const double *G = c->geo;
    const size_t P = (size_t)c->plane;
    g.Jo = G;
    g.Jx = G + P;
    g.Jy = G + 2 * P;
    g.Jq = G + 3 * P;
    g.Qi12o = G + 4 * P;
    g.Qi11x = G + 5 * P;
    g.Qi22y = G + 6 * P;
    g.JQo = G + 7 * P;
    g.fo = G + 8 * P;
    g.hs = c->hs;
    g.vsrc = c->vsrc;
    g.fsrc = c->fsrc;
    g.osrc = c->osrc;
    g.qnb = c->qnb;
    g.vsg = c->vsg;
    g.fsg = c->fsg;
    g.N = c->N;
    g.pitch = c->pitch;
    g.nbx = (c->N + 1 + swmc::BX - 1) / swmc::BX;
    g.nby = (c->N + 1 + swmc::BY - 1) / swmc::BY;
    g.ntiles = g.nbx * g.nby * 6;
    g.per = (g.ntiles + 7) / 8;
    g.plane = c->plane;
    g.fs = c->fs;
    g.hx = c->hx;
    g.scale = c->scale;
    g.grav = c->grav;
    g.dx1 = 1.0 / (c->scale * c->hx);
    return g;
}

// operator_swm_t%apply on the C grid for the input y (h, u, v), two launches; the tendencies go
// where RKM says
template <int RKM>
int c_enqueue_rhs(swm_cctx *c, const double *y, const swmc::RkArgs &r) {
    using K = swmc::Tiles;
    const swmc::CGeo g = make_cgeo(c);
    const swm::TileOrder o = K::order(c->N);
    const dim3 blk(K::THREADS), grd(o.blocks());
    hipLaunchKernelGGL(swmc::k_flux, grd, blk, 0, c->stream, o, g, y, c->wf(CW_G), c->wf(CW_KE), c->wf(CW_W));
    hipLaunchKernelGGL(swmc::k_tend<RKM>, grd, blk, 0, c->stream, o, g, y, c->wf(CW_G), c->wf(CW_KE), c->wf(CW_W), r);
    HIP_TRY(hipGetLastError());
    return SWM_OK;
}

// rk4_t%step (rk4_mod.f90:20-42): stage inputs state -> yA -> yB -> yA, the stage updates inside the
// tendency kernel; no stage writes a buffer that it reads at other points
int c_enqueue_rk4_step(swm_cctx *c, double *state, double dt) {
    const double c1 = 0.5 * dt, c2 = dt / 6.0, c3 = dt / 3.0;
    double *acc = c->wf(CW_ACC), *yA = c->wf(CW_YA), *yB = c->wf(CW_YB);
    int rc;
    if ((rc = c_enqueue_rhs<swmc::RK_S1>(c, state, {yA, state, acc, c1, c2}))) return rc;
    if ((rc = c_enqueue_rhs<swmc::RK_S23>(c, yA, {yB, state, acc, c1, c3}))) return rc;
    if ((rc = c_enqueue_rhs<swmc::RK_S23>(c, yB, {yA, state, acc, dt, c3}))) return rc;
    return c_enqueue_rhs<swmc::RK_S4>(c, yA, {state, nullptr, acc, 0.0, c2});
}

void c_drop_graphs(swm_cctx *c) {
    c->graphs.drop();
    c->graph_state = nullptr;
}

void c_free(swm_cctx *c) {
    if (!c) return;
    c_drop_graphs(c);
    for (void *p : {(void *)c->geo, (void *)c->hs, (void *)c->lists, (void *)c->signs, (void *)c->work, (void *)c->qw,
                    (void *)c->dpart, (void *)c->ecs_src, (void *)c->ecs_sign,
                    (void *)c->ecs_strips, (void *)c->ecs_ow, (void *)c->ecs_oind, (void *)c->ecs_vt,
                    (void *)c->ecs_vti, (void *)c->ecs_ext})
        if (p) (void)hipFree(p);
    if (c->own_stream && c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

// host <-> device copy of one field of point type t (nx x ny points) between the host tile layout
// (6, N+1+2hw, N+1+2hw) and the stored layout
int c_copy_field(swm_cctx *c, int t, double *dev, double *host, int hw, bool upload) {
    const int N = c->N, nx = N + (t == 1 || t == 3), ny = N + (t == 2 || t == 3), ld = N + 1 + 2 * hw;
    std::vector<double> buf((size_t)c->fs, 0.0);
    if (upload) {
        for (int p = 0; p < 6; ++p)
            for (int j = 1; j <= ny; ++j)
                for (int i = 1; i <= nx; ++i)
                    buf[((size_t)p * c->rows + (j - 1 + swmc::H)) * c->pitch + (i - 1 + swmc::H)] =
                        host[((size_t)p * ld + (j - 1 + hw)) * ld + (i - 1 + hw)];
        HIP_TRY(hipMemcpyAsync(dev, buf.data(), c->field_bytes(), hipMemcpyHostToDevice, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
    } else {
        HIP_TRY(hipMemcpyAsync(buf.data(), dev, c->field_bytes(), hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
        std::fill(host, host + (size_t)6 * ld * ld, 0.0);
        for (int p = 0; p < 6; ++p)
            for (int j = 1; j <= ny; ++j)
                for (int i = 1; i <= nx; ++i)
                    host[((size_t)p * ld + (j - 1 + hw)) * ld + (i - 1 + hw)] =
                        buf[((size_t)p * c->rows + (j - 1 + swmc::H)) * c->pitch + (i - 1 + swmc::H)];
    }
    return SWM_OK;
}

}  // namespace

extern "C" int swm_c_create(swm_cctx **out, int N, const char *div, const char *grad, const char *curl,
                            const char *coriolis, const char *ke, const char *co2contra, const char *massflux,
                            const char *quad, double scale, double omega, double grav) {
    if (!out) return fail(SWM_EARG, "ctx pointer is NULL");
    *out = nullptr;
    if (N < 8 || N > 8192) return fail(SWM_EARG, "N must be in [8, 8192]");
    if (!(scale > 0) || !(grav > 0)) return fail(SWM_EARG, "scale and grav must be positive");
    const std::pair<const char *, const char *> names[] = {
        {div, "divergence_c_sbp42"}, {grad, "gradient_c_sbp42"}, {curl, "curl_c_sbp42"},
        {coriolis, "coriolis_Cgrid_sbp42"}, {ke, "KE_Cgrid_sbp42"}, {co2contra, "co2contra_c_sbp42"},
        {massflux, "massflux_c_sbp42"}, {quad, "SBP_C42_quadrature"}};
    for (const auto &nm : names)
        if (!nm.first || std::string(nm.first) != nm.second)
            return fail(SWM_ENAME, std::string("unsupported C-grid operator name: ") + (nm.first ? nm.first : "(null)") +
                                       " (expected " + nm.second + ")");
    swm_cctx *c = new swm_cctx();
    c->N = N;
    c->rows = N + 1 + 2 * swmc::H;
    c->pitch = (c->rows + 7) / 8 * 8;
    c->plane = (long long)c->rows * c->pitch;
    c->fs = 6LL * c->plane;
    c->scale = scale;
    c->omega = omega;
    c->grav = grav;
    c->hx = (0.25 * std::acos(-1.0) - (-0.25 * std::acos(-1.0))) / (double)N;
    auto bail = [&](int code) { c_free(c); return code; };
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(SWM_EHIP, "hipStreamCreate failed"));
    c->own_stream = true;

    const size_t F = (size_t)c->fs;
    std::vector<double> geo(8 * F, 0.0);
    const double axis[3] = {0.0, 0.0, 1.0};
    double *G = geo.data();
    swmh_c_geometry(N, 0, swmc::H, c->rows, c->pitch, omega, axis, G, nullptr, G + 4 * F, nullptr, G + 7 * F);
    swmh_c_geometry(N, 1, swmc::H, c->rows, c->pitch, omega, axis, G + F, G + 5 * F, nullptr, nullptr, nullptr);
    swmh_c_geometry(N, 2, swmc::H, c->rows, c->pitch, omega, axis, G + 2 * F, nullptr, nullptr, G + 6 * F, nullptr);
    swmh_c_geometry(N, 3, swmc::H, c->rows, c->pitch, omega, axis, G + 3 * F, nullptr, nullptr, nullptr, nullptr);
    // device copy: panel 0 of the seven metric planes (every panel holds the same values, checked
    // here bit for bit), the product J Qi12 at o points, then f on all six panels
    const size_t P = (size_t)c->plane;
    std::vector<double> dgeo(8 * P + F);
    for (int w = 0; w < 7; ++w) {
        const double *m = G + (size_t)w * F;
        for (int p = 1; p < 6; ++p)
            if (std::memcmp(m, m + p * P, P * sizeof(double)) != 0)
                return bail(fail(SWM_EARG, "C-grid metric differs between panels"));
        std::copy(m, m + P, dgeo.begin() + (size_t)w * P);
    }
    for (size_t k = 0; k < P; ++k) dgeo[7 * P + k] = dgeo[k] * dgeo[4 * P + k];
    std::copy(G + 7 * F, G + 8 * F, dgeo.begin() + 8 * P);
    if (hipMalloc((void **)&c->geo, dgeo.size() * sizeof(double)) != hipSuccess ||
        hipMemcpy(c->geo, dgeo.data(), dgeo.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess)
        return bail(fail(SWM_EHIP, "C-grid geometry upload failed"));

    const int dvec = 3, dO = 3;
    const size_t mv = (size_t)6 * 4 * (N + 1) * dvec, mf = (size_t)6 * 4 * N, mo = (size_t)6 * 4 * N * dO,
                 mq = (size_t)6 * 4 * (N + 1);
    std::vector<long long> vd(mv), vs(mv), fd(mf), fsrc(mf), od(mo), os(mo), qo(mq), qn(mq);
    std::vector<signed char> vsg(mv), fsg(mf);
    int counts[4] = {0, 0, 0, 0};
    const int hr = swmh_c_halo_lists(N, swmc::H, c->rows, c->pitch, c->fs, dvec, dO, vd.data(), vs.data(), vsg.data(),
                                     fd.data(), fsrc.data(), fsg.data(), od.data(), os.data(), qo.data(), qn.data(), counts);
    if (hr != 0 || (size_t)counts[0] != mv || (size_t)counts[1] != mf || (size_t)counts[2] != mo || (size_t)counts[3] != mq)
        return bail(fail(SWM_EARG, "C-grid halo lists do not match the cube topology"));
    // every offset stays inside one field pair (the pair for vectors, one field otherwise)
    for (size_t k = 0; k < mv; ++k)
        if (vd[k] < 0 || vd[k] >= 2 * c->fs || vs[k] < 0 || vs[k] >= 2 * c->fs) return bail(fail(SWM_EARG, "vector halo offset out of range"));
    for (size_t k = 0; k < mf; ++k)
        if (fd[k] < 0 || fd[k] >= 2 * c->fs || fsrc[k] < 0 || fsrc[k] >= 2 * c->fs) return bail(fail(SWM_EARG, "face halo offset out of range"));
    for (size_t k = 0; k < mo; ++k)
        if (od[k] < 0 || od[k] >= c->fs || os[k] < 0 || os[k] >= c->fs) return bail(fail(SWM_EARG, "O halo offset out of range"));
    for (size_t k = 0; k < mq; ++k)
        if (qn[k] < 0 || qn[k] >= c->fs) return bail(fail(SWM_EARG, "q sync offset out of range"));
    // device lists: sources in the order the kernels index them (swmc::CGeo)
    std::vector<long long> L;
    L.reserve(mv + mf + mo + mq);
    for (auto *v : {&vs, &fsrc, &os, &qn}) L.insert(L.end(), v->begin(), v->end());
    std::vector<signed char> S;
    S.insert(S.end(), vsg.begin(), vsg.end());
    S.insert(S.end(), fsg.begin(), fsg.end());
    if (hipMalloc((void **)&c->lists, L.size() * sizeof(long long)) != hipSuccess ||
        hipMemcpy(c->lists, L.data(), L.size() * sizeof(long long), hipMemcpyHostToDevice) != hipSuccess ||
        hipMalloc((void **)&c->signs, S.size()) != hipSuccess ||
        hipMemcpy(c->signs, S.data(), S.size(), hipMemcpyHostToDevice) != hipSuccess)
        return bail(fail(SWM_EHIP, "C-grid halo list upload failed"));
    c->vsrc = c->lists;
    c->fsrc = c->vsrc + mv;
    c->osrc = c->fsrc + mf;
    c->qnb = c->osrc + mo;
    c->vsg = c->signs;
    c->fsg = c->signs + mv;
    {
        // create_mass_coefficients (quadrature_factory_mod.f90:156-175): A_centers (13/12, 7/8,
        // 25/24, 1, ...) and A_interfaces (7/18, 9/8, 1, 71/72, 1, ...) from both ends
        const double Ac[4] = {13.0 / 12.0, 7.0 / 8.0, 25.0 / 24.0, 1.0};
        const double Ai[5] = {7.0 / 18.0, 9.0 / 8.0, 1.0, 71.0 / 72.0, 1.0};
        std::vector<double> q((size_t)2 * (N + 2), 1.0);
        double *acen = q.data(), *aint = q.data() + (N + 2);
        for (int i = 1; i <= std::min(4, N); ++i) acen[i] = Ac[i - 1];
        for (int i = std::max(N - 3, 1); i <= N; ++i) acen[i] = Ac[N - i];
        for (int i = 1; i <= std::min(5, N + 1); ++i) aint[i] = Ai[i - 1];
        for (int i = std::max(N + 1 - 4, 1); i <= N + 1; ++i) aint[i] = Ai[N + 1 - i];
        c->dblocks = (long long)((N + 1 + swmc::BX - 1) / swmc::BX) * ((N + 1 + swmc::BY - 1) / swmc::BY) * 6;
        if (hipMalloc((void **)&c->qw, q.size() * sizeof(double)) != hipSuccess ||
            hipMemcpy(c->qw, q.data(), q.size() * sizeof(double), hipMemcpyHostToDevice) != hipSuccess ||
            hipMalloc((void **)&c->dpart, (size_t)(c->dblocks * 10 + 8) * sizeof(double)) != hipSuccess)
            return bail(fail(SWM_EHIP, "C-grid diagnostics set-up failed"));
    }
    const size_t wb = (size_t)CW_COUNT * c->field_bytes();
    if (hipMalloc((void **)&c->work, wb) != hipSuccess || hipMemset(c->work, 0, wb) != hipSuccess)
        return bail(fail(SWM_EHIP, "C-grid work buffer allocation failed"));
    if (hipDeviceSynchronize() != hipSuccess) return bail(fail(SWM_EHIP, "set-up synchronisation failed"));
    *out = c;
    return SWM_OK;
}

extern "C" int swm_c_destroy(swm_cctx *c) {
    if (!c) return fail(SWM_EARG, "ctx is NULL");
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    c_free(c);
    return SWM_OK;
}

extern "C" int swm_c_info(const swm_cctx *c, int *N, int *halo, int *rows, int *pitch, long long *field_elems) {
    if (!c) return fail(SWM_EARG, "ctx is NULL");
    if (N) *N = c->N;
    if (halo) *halo = swmc::H;
    if (rows) *rows = c->rows;
    if (pitch) *pitch = c->pitch;
    if (field_elems) *field_elems = c->fs;
    return SWM_OK;
}

extern "C" int swm_c_synchronize(swm_cctx *c) {
    if (!c) return fail(SWM_EARG, "ctx is NULL");
    HIP_TRY(hipStreamSynchronize(c->stream));
    return SWM_OK;
}

extern "C" int swm_c_state_alloc(swm_cctx *c, void **state) {
    if (!c || !state) return fail(SWM_EARG, "NULL argument");
    const size_t sb = 3 * c->field_bytes();
    HIP_TRY(hipMalloc(state, sb));
    HIP_TRY(hipMemsetAsync(*state, 0, sb, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    return SWM_OK;
}

extern "C" int swm_c_state_free(swm_cctx *c, void *state) {
    if (!c) return fail(SWM_EARG, "ctx is NULL");
    if (!state) return SWM_OK;
    HIP_TRY(hipStreamSynchronize(c->stream));
    if (c->graph_state == state) c_drop_graphs(c);
    HIP_TRY(hipFree(state));
    return SWM_OK;
}

extern "C" int swm_c_state_upload(swm_cctx *c, void *state, const double *h, const double *u, const double *v, int hw) {
    if (!c || !state || !h || !u || !v) return fail(SWM_EARG, "NULL argument");
    if (hw < 0 || hw > 64) return fail(SWM_EARG, "halo_width out of range");
    const double *src[3] = {h, u, v};
    for (int k = 0; k < 3; ++k) {
        int rc = c_copy_field(c, k, (double *)state + (size_t)k * c->fs, const_cast<double *>(src[k]), hw, true);
        if (rc) return rc;
    }
    return SWM_OK;
}

extern "C" int swm_c_state_download(swm_cctx *c, const void *state, double *h, double *u, double *v, int hw) {
    if (!c || !state || !h || !u || !v) return fail(SWM_EARG, "NULL argument");
    if (hw < 0 || hw > 64) return fail(SWM_EARG, "halo_width out of range");
    double *dst[3] = {h, u, v};
    for (int k = 0; k < 3; ++k) {
        int rc = c_copy_field(c, k, (double *)state + (size_t)k * c->fs, dst[k], hw, false);
        if (rc) return rc;
    }
    return SWM_OK;
}

extern "C" int swm_c_set_orography(swm_cctx *c, const double *hs, int hw) {
    if (!c) return fail(SWM_EARG, "ctx is NULL");
    if (hw < 0 || hw > 64) return fail(SWM_EARG, "halo_width out of range");
    HIP_TRY(hipStreamSynchronize(c->stream));
    c_drop_graphs(c);
    if (!hs) {
        if (c->hs) HIP_TRY(hipFree(c->hs));
        c->hs = nullptr;
        return SWM_OK;
    }
    if (!c->hs) {
        HIP_TRY(hipMalloc((void **)&c->hs, c->field_bytes()));
        HIP_TRY(hipMemsetAsync(c->hs, 0, c->field_bytes(), c->stream));
    }
    return c_copy_field(c, 0, c->hs, const_cast<double *>(hs), hw, true);
}

extern "C" int swm_c_rhs(swm_cctx *c, const void *vin, void *vout) {
    if (!c || !vin || !vout) return fail(SWM_EARG, "NULL argument");
    if (vin == vout) return fail(SWM_EARG, "vin and vout must differ");
    return c_enqueue_rhs<swmc::RK_RHS>(c, (const double *)vin, {(double *)vout, nullptr, nullptr, 0.0, 0.0});
}

extern "C" int swm_c_rk4_steps(swm_cctx *c, void *state, double dt, int nsteps) {
    if (!c || !state) return fail(SWM_EARG, "NULL argument");
    if (nsteps < 0) return fail(SWM_EARG, "nsteps must be >= 0");
    if (nsteps == 0) return SWM_OK;
    if (c->graph_state != state || c->graph_dt != dt) c_drop_graphs(c);
    c->graph_state = state;
    c->graph_dt = dt;
    return c->graphs.run(c->stream, 6LL * c->N * c->N, nsteps, [&] { return c_enqueue_rk4_step(c, (double *)state, dt); });
}

extern "C" int swm_c_diagnostics(swm_cctx *c, const void *state, double out[7]) {
    if (!c || !state || !out) return fail(SWM_EARG, "NULL argument");
    const swmc::CGeo g = make_cgeo(c);
    const dim3 blk(swmc::BX, swmc::BY), grd(8 * g.per);
    double *res = c->dpart + c->dblocks * 10;
    hipLaunchKernelGGL(swmc::k_cdiag_partial, grd, blk, 0, c->stream, g, (const double *)state, c->qw,
                       c->qw + (c->N + 2), c->dpart);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(swmc::k_cdiag_final, dim3(1), dim3(swm::FINAL_THREADS), 0, c->stream, c->dpart, c->dblocks, res);
    HIP_TRY(hipGetLastError());
    double r[6];
    HIP_TRY(hipMemcpyAsync(r, res, sizeof(r), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    const double ke = r[1] + r[2];
    out[0] = r[4];
    out[1] = r[5];
    out[2] = r[0];
    out[3] = ke + r[3];
    out[4] = ke;
    out[5] = r[3];
    out[6] = std::nan("");
    return SWM_OK;
}
