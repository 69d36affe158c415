// Hyperdiffusion of the Ah state with the narrow-stencil SBP Laplacians sbp21, sbp42 and sbp63,
// FP64 (sbp21: three-point rows, laplace_Ah_sbp21_narrow_mod.f90).
//
// Laplacian, laplace_Ah_sbp42_narrow_t%calc_laplace (differential_operators/horizontal/
// laplace/laplace_Ah_sbp42_narrow_mod.f90:23-763) and laplace_Ah_sbp63_narrow_t%calc_laplace
// (laplace_Ah_sbp63_narrow_mod.f90:494-1717), the same steps with their own tables:
//   d1x = Dx(f) J Qi12,  d1y = Dy(f) J Qi12                      (first-derivative SBP d42 / d63)
//   d2x = D2x(Qi11 J) f, d2y = D2y(Qi22 J) f                     (narrow variable-coefficient D2)
//   d2x -= 0.5 * pc * (-+2 d1y) on the x edges, then (-+2 d1x) on the y edges
//        (pc = 48/17 for sbp42, 43200/13649 for sbp63)
//   L f = ((d2x + d2y) + Dx(d1y) + Dy(d1x)) / (hx a)^2 / J, then the scalar edge sync.
// Hyperdiffusion of one field, hordiff_scalar_t%calc_diff (hordiff/hordiff_scalar_mod.f90:
// 34-59): tend = -(c a hx)^4 L(L f).  Velocity, hordiff_colocated_xyz_t%calc_diff_vec
// (hordiff/hordiff_colocated_mod.f90:39-58): Cartesian components V = b1 u + b2 v, the scalar
// hyperdiffusion of each, back as (V.b1, V.b2), covariant vector edge sync.
// Step, operator_swm_diff_t%apply + explicit_Eul1 (operator_swm_diff_mod.f90:25-46,
// time_schemes/explicit_Eul1_mod.f90:20-30): y += dt * tend.
//
// One step is three launches.  hd_lap (STEP 1) forms h and the Cartesian velocity from the state as it
// loads its tiles and writes their Laplacians; hd_lap (STEP 2) applies the edge sync as it reads them,
// forms the second Laplacian and, at the points off the panel edges, the tendencies and the Euler step;
// hd_edges does the panel-edge points.  Panel-edge results go to compact edge buffers, so that no
// kernel reads a value another block of the same launch overwrites.  swm_laplace is hd_lap (STEP 0) and
// hd_sync.
//
// A tile runs all its fields together.  The D2 weights depend on the metric only and are formed once per
// context (hd_weights) with the operations of the reference; a thread loads those of its point once and
// applies them to every field, as it does its indices and its metric terms.

#include <algorithm>
#include <type_traits>
#include <utility>

#include "swm_ctx.h"

#include "laplace_sbp42_narrow.h"
#include "laplace_sbp63_narrow.h"

namespace swm {

// The generated coefficient tables of one narrow Laplacian family, bound by name.
template <int ORD> struct Ln;
template <> struct Ln<42> {
    static constexpr int NB = LN42_NB, NCOL = LN42_NCOL, R = LN42_R;
    static constexpr bool NEG_INV_H = LN42_ROW_NEG_INV_H != 0;
    static constexpr auto &H = LN42_H;
    static constexpr auto &NCOLS = LN42_NCOLS;
    static constexpr auto &MSTART = LN42_MSTART;
    static constexpr auto &TCOEF = LN42_TCOEF;
    static constexpr auto &TSIGN = LN42_TSIGN;
    static constexpr auto &TB = LN42_TB;
    static constexpr auto &ISTART = LN42_ISTART;
    static constexpr auto &ICOEF = LN42_ICOEF;
    static constexpr auto &ISIGN = LN42_ISIGN;
    static constexpr auto &IB = LN42_IB;
    static constexpr double PC = LN42_PC;
};
template <> struct Ln<63> {
    static constexpr int NB = LN63_NB, NCOL = LN63_NCOL, R = LN63_R;
    static constexpr bool NEG_INV_H = LN63_ROW_NEG_INV_H != 0;
    static constexpr auto &H = LN63_H;
    static constexpr auto &NCOLS = LN63_NCOLS;
    static constexpr auto &MSTART = LN63_MSTART;
    static constexpr auto &TCOEF = LN63_TCOEF;
    static constexpr auto &TSIGN = LN63_TSIGN;
    static constexpr auto &TB = LN63_TB;
    static constexpr auto &ISTART = LN63_ISTART;
    static constexpr auto &ICOEF = LN63_ICOEF;
    static constexpr auto &ISIGN = LN63_ISIGN;
    static constexpr auto &IB = LN63_IB;
    static constexpr double PC = LN63_PC;
};

// sbp21: edge rows -(b0+b1) f0 + (b0+b1) f1, interior (bp+bc)/2 f+ - (bm+2bc+bp)/2 f + (bm+bc)/2 f-, summed
// in this order (from the right neighbour)
template <> struct Ln<21> {
    static constexpr int NB = 1, NCOL = 2, R = 1;
    static constexpr bool NEG_INV_H = false;
    static constexpr double H[1] = {1.0};
    static constexpr int NCOLS[1] = {2};
    static constexpr double PC = 2.0;
};

// Basis vectors b1, b2 of the panels: panel 0's give three prototype components, the first without b2, the
// second without b1; every panel's Cartesian components are the prototype's, permuted and signed
// (checked at set-up), so four planes of one panel serve all.  perm[8 p + k]: Cartesian component of
// prototype component k on panel p; perm[8 p + 4 + k]: its sign.
struct HdGeo {
    const double *J, *Qi11, *Qi12, *Qi22;   // panel 0 serves all panels if mps = 0
    const double *B0, *B1, *B2a, *B2b;      // b1 of component 0, b2 of component 1, b1 and b2 of component 2
    const int *perm;
    // per panel-edge slot: (slot of the neighbour's copy across the x edge or -1, across the y edge or -1,
    // their component codes), the weights of the vector sync along x and y edges, and b1, b2 (6 planes)
    const int4 *et;
    const double *eq, *eb;
    int n, pitch, es;
    long long fs, mps;
    double hs2;                             // (hx * scale)^2
};

// D2 weights of one family: interior planes (2R+1 per direction, point (i, j) at j*pitch + i), closure rows
// (side, row, weight) by the position along the edge
struct HdLn {
    const double *ix, *iy, *cx, *cy;
};

__device__ __forceinline__ void slot_point(int n, int sl, int &i, int &j) {
    if (sl < n) { i = sl; j = 0; }
    else if (sl < 2 * n) { i = sl - n; j = n - 1; }
    else if (sl < 3 * n - 2) { i = 0; j = sl - 2 * n + 1; }
    else { i = n - 1; j = sl - (3 * n - 2) + 1; }
}

// Closure row RW of the narrow D2 with b[k], fv[c] taken k, c points from the panel edge, and
// the interior row, expanded at compile time (every index and weight a constant): each weight
// is the table's constant expression folded to a double, products and sums in table order.
template <int ORD, int T>
__device__ __forceinline__ double ln_term(const double *b) {
    constexpr double w = Ln<ORD>::TCOEF[T];
    return w * b[Ln<ORD>::TB[T]];
}
template <int ORD, int T0, int... Is>
__device__ __forceinline__ double ln_sum(const double *b, std::integer_sequence<int, Is...>) {
    using L = Ln<ORD>;
    double m = 0.0;
    ((m = Is == 0 ? (L::TSIGN[T0 + Is] < 0 ? -ln_term<ORD, T0 + Is>(b) : ln_term<ORD, T0 + Is>(b))
                  : (L::TSIGN[T0 + Is] < 0 ? m - ln_term<ORD, T0 + Is>(b) : m + ln_term<ORD, T0 + Is>(b))),
     ...);
    return m;
}
template <int ORD, int RW, int C>
__device__ __forceinline__ double ln_m(const double *b) {
    using L = Ln<ORD>;
    constexpr int t0 = L::MSTART[RW][C], cnt = L::MSTART[RW][C + 1] - L::MSTART[RW][C];
    return ln_sum<ORD, t0>(b, std::make_integer_sequence<int, cnt>{});
}
template <int ORD, int T>
__device__ __forceinline__ double ln_iterm(const double *b) {
    constexpr double w = Ln<ORD>::ICOEF[T];
    return w * b[Ln<ORD>::IB[T] + Ln<ORD>::R];
}
template <int ORD, int T0, int... Is>
__device__ __forceinline__ double ln_isum(const double *b, std::integer_sequence<int, Is...>) {
    using L = Ln<ORD>;
    double m = 0.0;
    ((m = Is == 0 ? (L::ISIGN[T0 + Is] < 0 ? -ln_iterm<ORD, T0 + Is>(b) : ln_iterm<ORD, T0 + Is>(b))
                  : (L::ISIGN[T0 + Is] < 0 ? m - ln_iterm<ORD, T0 + Is>(b) : m + ln_iterm<ORD, T0 + Is>(b))),
     ...);
    return m;
}
template <int ORD, int O>
__device__ __forceinline__ double ln_icoef(const double *b) {
    using L = Ln<ORD>;
    return ln_isum<ORD, L::ISTART[O]>(b, std::make_integer_sequence<int, L::ISTART[O + 1] - L::ISTART[O]>{});
}
// weights of the narrow D2 row t of a line of n points with coefficient b(a): closure rows (from the near
// edge) and interior rows (from t - R, sbp21 from t + R)
template <int ORD, int RW, int... Cs>
__device__ __forceinline__ void ln_row_weights(const double *b, double *w, std::integer_sequence<int, Cs...>) {
    ((w[Cs] = ln_m<ORD, RW, Cs>(b)), ...);
}
template <int ORD, int... RWs>
__device__ __forceinline__ void ln_closure_weights(int r, const double *b, double *w, std::integer_sequence<int, RWs...>) {
    ((r == RWs ? ln_row_weights<ORD, RWs>(b, w, std::make_integer_sequence<int, Ln<ORD>::NCOLS[RWs]>{}) : (void)0), ...);
}
template <int ORD, int... Os>
__device__ __forceinline__ void ln_interior_weights(const double *b, double *w, std::integer_sequence<int, Os...>) {
    ((w[Os] = ln_icoef<ORD, Os>(b)), ...);
}

// one thread per point: its D2 weights along x (blockIdx.y = 0) or y (1), b = Qi11 J or Qi22 J
template <int ORD>
__global__ void __launch_bounds__(256) hd_weights(HdGeo g, double *__restrict__ inner, double *__restrict__ closure) {
    using L = Ln<ORD>;
    const int n = g.n, t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n * n) return;
    const int i = t % n, j = t / n;
    const bool alongx = blockIdx.y == 0;
    const double *Q = alongx ? g.Qi11 : g.Qi22;
    const int k = alongx ? i : j, pos = alongx ? j : i;
    const long long plane = (long long)n * g.pitch;
    double *in = inner + (alongx ? 0 : (2 * L::R + 1) * plane), *cl = closure + (alongx ? 0 : 2 * L::NB * L::NCOL * n);
    auto b = [&](int a) {
        const long long o = alongx ? (long long)j * g.pitch + a : (long long)a * g.pitch + i;
        return Q[o] * g.J[o];
    };
    const bool left = k < L::NB, right = k >= n - L::NB;
    if (left || right) {
        const int r = left ? k : n - 1 - k;
        double bb[L::NCOL], w[L::NCOL];
        for (int q = 0; q < L::NCOL; ++q) {
            bb[q] = b(left ? q : n - 1 - q);
            w[q] = 0.0;
        }
        if constexpr (ORD == 21) {
            w[0] = -(bb[0] + bb[1]);
            w[1] = +(bb[0] + bb[1]);
        } else {
            ln_closure_weights<ORD>(r, bb, w, std::make_integer_sequence<int, L::NB>{});
        }
        for (int q = 0; q < L::NCOL; ++q) cl[(((right ? L::NB : 0) + r) * L::NCOL + q) * n + pos] = w[q];
        return;
    }
    double bb[2 * L::R + 1], w[2 * L::R + 1];
    for (int q = 0; q < 2 * L::R + 1; ++q) bb[q] = b(k - L::R + q);
    if constexpr (ORD == 21) {
        w[0] = (bb[2] + bb[1]) / 2;
        w[1] = -(bb[0] + 2 * bb[1] + bb[2]) / 2;
        w[2] = (bb[0] + bb[1]) / 2;
    } else {
        ln_interior_weights<ORD>(bb, w, std::make_integer_sequence<int, 2 * L::R + 1>{});
    }
    for (int q = 0; q < 2 * L::R + 1; ++q) in[q * plane + (long long)j * g.pitch + i] = w[q];
}

// LDS of a tile of TX x TY points with NF fields: f on the box of lines its rows read (+-R points in the
// interior, points 0..NCOL-1 / n-NCOL..n-1 where it holds closure rows: the narrow D2 closure reads 2 /
// 8 / 12 points (sbp21 / 42 / 63), the first-derivative closure 2 / 6 / 9), the first derivatives
// d1y = Dy(f) J Qi12 on the tile rows and d1x = Dx(f) J Qi12 on the tile columns
template <int ORD, int TX, int TY>
struct HdTile {
    static constexpr int R = Ln<ORD>::R, B = Ln<ORD>::NB, NR = Ln<ORD>::NCOL;
    // the first-derivative operator of the family reads within the same box
    static_assert(-Sbp<ORD>::INSHIFT <= R && Sbp<ORD>::WIN + Sbp<ORD>::INSHIFT - 1 <= R, "d1 reach");
    static_assert(Sbp<ORD>::NE <= B && Sbp<ORD>::NW <= NR, "d1 closure");
    // box extent along a tile side of t points: interior rows give t + 2 R lines, closure rows at one
    // edge at most t + R + B - 1 (or NR); a tile holding closure rows of both edges (a0 < B, a0 a
    // multiple of t, and a0 + t > n - B) covers the whole line, n <= a0 + t + B - 1
    static constexpr int both(int t) { return ((B - 1) / t) * t + t + B - 1; }
    static constexpr int ext(int t) { return t + R + (R > B - 1 ? R : B - 1); }
    static constexpr int one(int t) { return ext(t) > NR ? ext(t) : NR; }
    static constexpr int span(int t) { return one(t) > both(t) ? one(t) : both(t); }
    static constexpr int LW = span(TX), LH = span(TY), NT = TX * TY;
    static constexpr int M = B > R ? B : R + 1;   // points between an inner tile and the panel edge
};
template <int W, int H, int TX, int TY, int NF>
struct HdSmem {
    double f[NF][H][W], dy[NF][TY][W], dx[NF][H][TX];
};

template <int ORD>
__device__ __forceinline__ void hd_rows(int a0, int ae, int n, int &lo, int &hi) {
    constexpr int R = Ln<ORD>::R, B = Ln<ORD>::NB, NR = Ln<ORD>::NCOL;
    lo = a0 - R > 0 ? a0 - R : 0;
    hi = ae + R < n ? ae + R : n;
    if (a0 < B) {
        lo = 0;
        const int m = NR < n ? NR : n;
        hi = hi > m ? hi : m;
    }
    if (ae > n - B) {
        hi = n;
        const int m = n - NR > 0 ? n - NR : 0;
        lo = lo < m ? lo : m;
    }
}

// scalar edge sync (halo_Ah_scalar_sync_mod.f90:52-93) of one field at a panel-edge slot: its raw value and
// those of its copies across the x edge (a) and the y edge (b)
__device__ __forceinline__ double hd_mean(bool ex, bool ey, double own, double a, double b) {
    if (ex && ey) return (own + a + b) / 3.0;
    return 0.5 * (own + (ex ? a : b));
}
__device__ __forceinline__ double hd_synced(const HdGeo &g, const double *__restrict__ E, int k, int sl) {
    const double *Ek = E + (long long)k * 6 * g.es;
    const int4 e = g.et[sl];
    return hd_mean(e.x >= 0, e.y >= 0, Ek[sl], e.x >= 0 ? Ek[e.x] : 0.0, e.y >= 0 ? Ek[e.y] : 0.0);
}

// Cartesian components of b1 and b2 on a panel from the prototype planes at a point
struct HdBasis {
    double b1[3], b2[3];
};
__device__ __forceinline__ HdBasis hd_basis(const HdGeo &g, int p, unsigned off) {
    const double v1[3] = {at_byte(g.B0, off), 0.0, at_byte(g.B2a, off)}, v2[3] = {0.0, at_byte(g.B1, off), at_byte(g.B2b, off)};
    HdBasis r{};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int c = g.perm[8 * p + k];
        const double s = g.perm[8 * p + 4 + k] < 0 ? -1.0 : 1.0;
#pragma unroll
        for (int q = 0; q < 3; ++q)
            if (q == c) {
                r.b1[q] = s * v1[k];
                r.b2[q] = s * v2[k];
            }
    }
    return r;
}

// final combination of hd_lap (STEP 2) and hd_edges: ht = ch L L h, (ut, vt) = (V.b1, V.b2) of
// V = cuv L L (Vx, Vy, Vz); yo = y0 + dt * tend (explicit_Eul1) or, with y0 = NULL, yo = tend
struct HdFin {
    const double *y0;
    double *yo;
    double ch, cuv, dt;
};

// One tile of hd_lap, fields h (H) and / or Vx, Vy, Vz (UV): STEP 0 the field h from `in` to `out`, STEP 1 from
// the state `in` to the work fields `out`, STEP 2 from the work fields `in` (panel edges: synced from Ein)
// to the state of `fin`.  Panel-edge results go to Eout.  INNER: the tile holds no closure row and its box, the
// tile +-R, no panel-edge point, so every row of it is an interior row.
// Bound by latency with three blocks a CU (LDS 41 KB at sbp42, 96 and 115 registers): its waves wait 57 % of
// their cycles, its vector instructions need 15 us and its fields at the rate of a large copy 10 us of the
// 39 (STEP 1) and 42 us (STEP 2) at C384 sbp42, alone on the chip (45 and 56 in plain band order); C191 sbp63:
// 23 and 28 us (27 and 33).  The six separate launches of the four fields that they take the place of took 167 us and 85 us with the edge launches.
template <int ORD, bool H, bool UV, int STEP, int TX, int TY, bool INNER, class Smem>
__device__ __forceinline__ void hd_lap_run(const HdGeo &g, const HdLn &ln, const double *__restrict__ in, double *__restrict__ out,
                                           const double *__restrict__ Ein, double *__restrict__ Eout, const HdFin &fin,
                                           int p, int x0, int y0, Smem &sm, double *tab) {
    using C = HdTile<ORD, TX, TY>;
    using L = Ln<ORD>;
    constexpr int NF = (H ? 1 : 0) + (UV ? 3 : 0), K0 = H ? 0 : 1, NT = C::NT, R = C::R;
    constexpr int BW = INNER ? TX + 2 * R : C::LW, BH = INNER ? TY + 2 * R : C::LH;
    constexpr int PB = (BW * BH + NT - 1) / NT, P1 = (BW * TY + NT - 1) / NT, P2 = (TX * BH + NT - 1) / NT;
    const int n = g.n, pitch = g.pitch, tid = threadIdx.x;
    const int xe = INNER ? x0 + TX : (x0 + TX < n ? x0 + TX : n), ye = INNER ? y0 + TY : (y0 + TY < n ? y0 + TY : n);
    int lx = x0 - R, hx = xe + R, ly = y0 - R, hy = ye + R;
    if constexpr (!INNER) {
        hd_rows<ORD>(x0, xe, n, lx, hx);
        hd_rows<ORD>(y0, ye, n, ly, hy);
    }
    const long long pb = (long long)p * n * pitch, mb = (long long)p * g.mps;
    const double *J = g.J + mb, *Q12 = g.Qi12 + mb;
    auto off = [&](int i, int j) { return (__umul24((unsigned)j, (unsigned)pitch) + (unsigned)i) * 8u; };
    // points of the box (kind 0), of the tile rows on the box's columns (1), of the box's rows on the tile
    // columns (2)
    auto box = [&](int q, int &c, int &r) { r = q / BW; c = q - r * BW; return INNER ? q < BW * BH : r < hy - ly && c < hx - lx; };
    auto row = [&](int q, int &c, int &r) { r = q / BW; c = q - r * BW; return INNER ? q < BW * TY : r < ye - y0 && c < hx - lx; };
    auto col = [&](int q, int &c, int &r) { r = q / TX; c = q - r * TX; return INNER ? q < TX * BH : r < hy - ly && c < xe - x0; };

    // ---- loads: the fields on the box, J and Qi12 where the first derivatives are formed ----
    double fv[PB][NF];
    double j1[P1], q1[P1], j2[P2], q2[P2];
#pragma unroll
    for (int k = 0; k < PB; ++k) {
        int c, r;
        if (!box(tid + k * NT, c, r)) continue;
        const int i = lx + c, j = ly + r;
        const unsigned o = off(i, j);
        if constexpr (STEP == 0) {
            fv[k][0] = at_byte(in + pb, o);
        } else if constexpr (STEP == 1) {
            if constexpr (H) fv[k][0] = at_byte(in + pb, o);
            if constexpr (UV) {
                // V = b1 u + b2 v (vec_math_mod.f90:107-126), prototype components
                const double u = at_byte(in + (g.fs + pb), o), v = at_byte(in + (2 * g.fs + pb), o);
                fv[k][NF - 3] = at_byte(g.B0, o) * u + 0.0 * v;
                fv[k][NF - 2] = 0.0 * u + at_byte(g.B1, o) * v;
                fv[k][NF - 1] = at_byte(g.B2a, o) * u + at_byte(g.B2b, o) * v;
            }
        } else {
            const bool edge = !INNER && (i == 0 || j == 0 || i == n - 1 || j == n - 1);
            const int sl = edge ? p * g.es + edge_slot(n, i, j) : 0;
#pragma unroll
            for (int l = 0; l < NF; ++l)
                fv[k][l] = edge ? hd_synced(g, Ein, K0 + l, sl) : at_byte(in + ((K0 + l) * g.fs + pb), o);
        }
    }
#pragma unroll
    for (int k = 0; k < P1; ++k) {
        int c, r;
        if (!row(tid + k * NT, c, r)) continue;
        const unsigned o = off(lx + c, y0 + r);
        j1[k] = at_byte(J, o);
        q1[k] = at_byte(Q12, o);
    }
#pragma unroll
    for (int k = 0; k < P2; ++k) {
        int c, r;
        if (!col(tid + k * NT, c, r)) continue;
        const unsigned o = off(x0 + c, ly + r);
        j2[k] = at_byte(J, o);
        q2[k] = at_byte(Q12, o);
    }
    if constexpr (!INNER)
        for (int c = tid; c < RowWeights<ORD>::SIZE; c += NT) tab[c] = row_weights<ORD>.w[c];
    // LDS field and sign of the loaded components
    int slot[NF];
    double sg[NF];
#pragma unroll
    for (int l = 0; l < NF; ++l) {
        slot[l] = l;
        sg[l] = 1.0;
        if (STEP == 1 && UV && l >= NF - 3) {
            slot[l] = NF - 3 + g.perm[8 * p + l - (NF - 3)];
            sg[l] = g.perm[8 * p + 4 + l - (NF - 3)] < 0 ? -1.0 : 1.0;
        }
    }
#pragma unroll
    for (int k = 0; k < PB; ++k) {
        int c, r;
        if (!box(tid + k * NT, c, r)) continue;
#pragma unroll
        for (int l = 0; l < NF; ++l) sm.f[slot[l]][r][c] = sg[l] * fv[k][l];
    }
    __syncthreads();

    // ---- first derivatives at the cross positions (calc_tile_d1x_d1y: sbp42 :60-93, sbp63 :531-564); the
    // own point's D2 weights and J, and what the Euler step reads, are loaded meanwhile ----
    const int tx = tid % TX, ty = tid / TX, i = x0 + tx, j = y0 + ty;
    const bool own = INNER || (i < n && j < n);
    constexpr int NI = 2 * R + 1, NW = INNER ? NI : (L::NCOL > NI ? L::NCOL : NI);
    constexpr bool REV = ORD == 21;   // interior rows summed from the right
    double wx[NW], wy[NW], Jo = 1.0, ihx = 1.0, ihy = 1.0;
    int bx = i + (REV ? R : -R), sx = REV ? -1 : 1, nx = NI, by = j + (REV ? R : -R), sy = sx, ny = NI;
    const unsigned oo = off(i, j);
    const long long plane = (long long)n * pitch;
    if (own) {
        Jo = at_byte(J, oo);
        bool inx = true, iny = true;
        if constexpr (!INNER) {
            inx = i >= L::NB && i < n - L::NB;
            iny = j >= L::NB && j < n - L::NB;
        }
        if (inx) {
#pragma unroll
            for (int q = 0; q < NI; ++q) wx[q] = at_byte(ln.ix + q * plane, oo);
        }
        if (iny) {
#pragma unroll
            for (int q = 0; q < NI; ++q) wy[q] = at_byte(ln.iy + q * plane, oo);
        }
        if constexpr (!INNER) {
            auto closure = [&](int t, int pos, const double *cl, double *w, int &b, int &s, int &cnt, double &ih) {
                const bool left = t < L::NB;
                const int rr = left ? t : n - 1 - t;
                b = left ? 0 : n - 1;
                s = left ? 1 : -1;
                cnt = 0;
#pragma unroll
                for (int q = 0; q < L::NB; ++q)
                    if (q == rr) {
                        cnt = L::NCOLS[q];
                        ih = 1.0 / L::H[q];
                    }
                const double *c0 = cl + (long long)((left ? 0 : L::NB) + rr) * L::NCOL * n + pos;
#pragma unroll
                for (int q = 0; q < L::NCOL; ++q) w[q] = c0[q * n];
            };
            if (!inx) closure(i, j, ln.cx, wx, bx, sx, nx, ihx);
            if (!iny) closure(j, i, ln.cy, wy, by, sy, ny, ihy);
        }
    }
    auto d1 = [&](int t, int lo, const auto &get) {     // get(local index)
        if constexpr (INNER) return sbp_row_in<ORD, double>(t - lo, get);
        else {
            const RowAt ra = row_at<ORD>(t, n);
            constexpr int RN = RowWeights<ORD>::NW;
            const double *w = tab + ra.cls * RN;
            double s = w[0] * get(ra.base - lo);
#pragma unroll
            for (int m = 1; m < RN; ++m)
                if (m < ra.cnt) s = s + w[m] * get(ra.base - lo + m);
            return s;
        }
    };
#pragma unroll
    for (int k = 0; k < P1; ++k) {
        int c, r;
        if (!row(tid + k * NT, c, r)) continue;
#pragma unroll
        for (int l = 0; l < NF; ++l) sm.dy[l][r][c] = d1(y0 + r, ly, [&](int q) { return sm.f[l][q][c]; }) * j1[k] * q1[k];
    }
#pragma unroll
    for (int k = 0; k < P2; ++k) {
        int c, r;
        if (!col(tid + k * NT, c, r)) continue;
#pragma unroll
        for (int l = 0; l < NF; ++l) sm.dx[l][r][c] = d1(x0 + c, lx, [&](int q) { return sm.f[l][r][q]; }) * j2[k] * q2[k];
    }
    double y0v[3] = {};
    HdBasis bs{};
    if constexpr (STEP == 2) {
        if (own) {
            if (UV) bs = hd_basis(g, p, oo);
            if (fin.y0) {
#pragma unroll
                for (int k = H ? 0 : 1; k < (UV ? 3 : 1); ++k) y0v[k] = at_byte(fin.y0 + (k * g.fs + pb), oo);
            }
        }
    }
    __syncthreads();
    if (!own) return;

    // ---- D2 rows, cross derivatives, penalties of the cross terms (sbp42 :716-742, sbp63 :1671-1697) ----
    const int cx = i - lx, cy = j - ly;
    auto d2 = [&](const double *w, int b, int s, int cnt, double ih, bool closure, const auto &get) {
        double v = w[0] * get(b);
        if constexpr (INNER) {
#pragma unroll
            for (int q = 1; q < NI; ++q) v = v + w[q] * get(b + s * q);
            return v;
        } else {
#pragma unroll
            for (int q = 1; q < NW; ++q)
                if (q < cnt) v = v + w[q] * get(b + s * q);
            if (L::NEG_INV_H && closure) v = -(ih * v);
            return v;
        }
    };
    const bool clx = !INNER && (i < L::NB || i >= n - L::NB), cly = !INNER && (j < L::NB || j >= n - L::NB);
    const bool edge = !INNER && (i == 0 || j == 0 || i == n - 1 || j == n - 1);
    double res[NF];
#pragma unroll
    for (int l = 0; l < NF; ++l) {
        double d2x = d2(wx, bx - lx, sx, nx, ihx, clx, [&](int q) { return sm.f[l][cy][q]; });
        const double d2y = d2(wy, by - ly, sy, ny, ihy, cly, [&](int q) { return sm.f[l][q][cx]; });
        if constexpr (!INNER) {
            constexpr double pc = L::PC;
            if (i == 0) d2x = d2x - 0.5 * (pc * (-2.0 * sm.dy[l][ty][cx]));
            if (i == n - 1) d2x = d2x - 0.5 * (pc * (2.0 * sm.dy[l][ty][cx]));
            if (j == 0) d2x = d2x - 0.5 * (pc * (-2.0 * sm.dx[l][cy][tx]));
            if (j == n - 1) d2x = d2x - 0.5 * (pc * (2.0 * sm.dx[l][cy][tx]));
        }
        const double d2yx = d1(j, ly, [&](int q) { return sm.dx[l][q][tx]; });
        const double d2xy = d1(i, lx, [&](int q) { return sm.dy[l][ty][q]; });
        double v = 1.0 * d2x + 1.0 * d2y;
        v = v + 1.0 * d2xy + 1.0 * d2yx;
        res[l] = v / g.hs2 / Jo;
    }
    if (edge) {
        const int sl = p * g.es + edge_slot(n, i, j);
#pragma unroll
        for (int l = 0; l < NF; ++l) Eout[(long long)(K0 + l) * 6 * g.es + sl] = res[l];
    } else if constexpr (STEP < 2) {
#pragma unroll
        for (int l = 0; l < NF; ++l) at_byte(out + ((K0 + l) * g.fs + pb), oo) = res[l];
    } else {
        if constexpr (H) {
            const double ht = fin.ch * res[0];
            at_byte(fin.yo + pb, oo) = fin.y0 ? y0v[0] + fin.dt * ht : ht;
        }
        if constexpr (UV) {
            const double Vx = fin.cuv * res[NF - 3], Vy = fin.cuv * res[NF - 2], Vz = fin.cuv * res[NF - 1];
            const double ut = Vx * bs.b1[0] + Vy * bs.b1[1] + Vz * bs.b1[2];
            const double vt = Vx * bs.b2[0] + Vy * bs.b2[1] + Vz * bs.b2[2];
            at_byte(fin.yo + (g.fs + pb), oo) = fin.y0 ? y0v[1] + fin.dt * ut : ut;
            at_byte(fin.yo + (2 * g.fs + pb), oo) = fin.y0 ? y0v[2] + fin.dt * vt : vt;
        }
    }
}

template <int ORD, bool H, bool UV, int STEP, int TX, int TY>
__global__ void __launch_bounds__(TX * TY) hd_lap(TileOrder order, HdGeo g, HdLn ln, const double *__restrict__ in, double *__restrict__ out,
                                                  const double *__restrict__ Ein, double *__restrict__ Eout, HdFin fin) {
    using C = HdTile<ORD, TX, TY>;
    constexpr int NF = (H ? 1 : 0) + (UV ? 3 : 0), R = C::R;
    __shared__ union { HdSmem<TX + 2 * R, TY + 2 * R, TX, TY, NF> in; HdSmem<C::LW, C::LH, TX, TY, NF> any; } sm;
    __shared__ double tab[RowWeights<ORD>::SIZE];
    const int n = g.n;
    const TilePos at = tile_pos(order, blockIdx.x);
    const int p = at.p, x0 = at.cx * TX, y0 = at.cy * TY;
    constexpr int M = C::M;
    if (x0 >= M && x0 + TX <= n - M && y0 >= M && y0 + TY <= n - M)
        hd_lap_run<ORD, H, UV, STEP, TX, TY, true>(g, ln, in, out, Ein, Eout, fin, p, x0, y0, sm.in, tab);
    else
        hd_lap_run<ORD, H, UV, STEP, TX, TY, false>(g, ln, in, out, Ein, Eout, fin, p, x0, y0, sm.any, tab);
}

// scalar edge sync of the raw edge values E of one field into out
__global__ void hd_sync(HdGeo g, const double *__restrict__ E, double *__restrict__ out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 6 * g.es) return;
    const int p = t / g.es;
    int i, j;
    slot_point(g.n, t - p * g.es, i, j);
    out[((long long)p * g.n + j) * g.pitch + i] = hd_synced(g, E, 0, t);
}

// The panel-edge points of a step from the raw second Laplacians E: scalar edge syncs, tendencies on
// every panel that holds the point, covariant vector edge sync of the velocity's (ecs_Ah_vec_sync_mod.f90:
// 51-124, components entering as (U, V) = (vt, ut)), final combination.  A few waves, bound by the chain of
// loads: the tables hold each slot's copies, sync weights and basis, so that it is table, edge values,
// stores (4.8 us at C384 and C191; 15 us walking the neighbour table and the basis planes).
__global__ void __launch_bounds__(64) hd_edges(HdGeo g, const double *__restrict__ E, HdFin fin) {
    const int ns = 6 * g.es;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= ns) return;
    const int4 e = g.et[t];
    const bool ex = e.x >= 0, ey = e.y >= 0, corner = ex && ey;
    const int sx = ex ? e.x : t, sy = ey ? e.y : t;
    double own[4], a[4], b[4], b0[6], ba[6], bb[6], y0v[3];
    const int p = t / g.es;
    int i, j;
    slot_point(g.n, t - p * g.es, i, j);
    const long long o = ((long long)p * g.n + j) * g.pitch + i;
#pragma unroll
    for (int k = 0; k < 4; ++k) own[k] = E[(long long)k * ns + t];
#pragma unroll
    for (int k = 0; k < 6; ++k) b0[k] = g.eb[(long long)k * ns + t];
#pragma unroll
    for (int k = 0; k < 3; ++k) y0v[k] = fin.y0 ? fin.y0[k * g.fs + o] : 0.0;
    const double qx = g.eq[t], qy = g.eq[ns + t];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        a[k] = E[(long long)k * ns + sx];
        b[k] = E[(long long)k * ns + sy];
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        ba[k] = g.eb[(long long)k * ns + sx];
        bb[k] = g.eb[(long long)k * ns + sy];
    }
    // at a cube corner the copies are those of this slot in another order
    const int4 ea = corner ? g.et[sx] : e, eb = corner ? g.et[sy] : e;
    auto value = [&](int k, int s) { return s == t ? own[k] : s == sx ? a[k] : b[k]; };
    double S[4], Sa[4], Sb[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        S[k] = hd_mean(ex, ey, own[k], a[k], b[k]);
        Sa[k] = corner ? (a[k] + value(k, ea.x) + value(k, ea.y)) / 3.0 : S[k];
        Sb[k] = corner ? (b[k] + value(k, eb.x) + value(k, eb.y)) / 3.0 : S[k];
    }
    auto uv = [&](const double *v, const double *w, double &ut, double &vt) {
        const double tx = fin.cuv * v[1], ty = fin.cuv * v[2], tz = fin.cuv * v[3];
        ut = tx * w[0] + ty * w[1] + tz * w[2];
        vt = tx * w[3] + ty * w[4] + tz * w[5];
    };
    double V, U, gx, gy, Vx, Ux, Vy, Uy, ut, vt;
    uv(S, b0, V, U);
    uv(Sa, ba, ut, vt);
    map_vec(e.z & 255, ut, vt, Vx, Ux);
    uv(Sb, bb, ut, vt);
    map_vec(e.z >> 8, ut, vt, Vy, Uy);
    if (corner) {
        gy = (U + Ux + Uy + qy * Vy) / 3.0;
        gx = (V + Vx + Vy + qx * Ux) / 3.0;
    } else if (ex) {
        gy = 0.5 * (U + Ux);
        gx = 0.5 * (V + Vx + qx * Ux);
    } else {
        gx = 0.5 * (V + Vy);
        gy = 0.5 * (U + Uy + qy * Vy);
    }
    const double tend[3] = {fin.ch * S[0], gx, gy};
#pragma unroll
    for (int k = 0; k < 3; ++k) fin.yo[k * g.fs + o] = fin.y0 ? y0v[k] + fin.dt * tend[k] : tend[k];
}

}  // namespace swm

// ------------------------------------------------------------------------------------------------
// Host side
namespace swm_host {

struct HdWork {
    double *basis = nullptr;                      // B0, B1, B2a, B2b: one panel plane each
    int *perm = nullptr;
    int4 *et = nullptr;                           // panel-edge tables (HdGeo): copies, sync weights, basis
    double *eq = nullptr, *eb = nullptr;
    double *W = nullptr;                          // first Laplacians of h, Vx, Vy, Vz
    double *E1 = nullptr, *E2 = nullptr;          // 4 x ns edge values each
    double *ln[3] = {nullptr, nullptr, nullptr};  // D2 weights of sbp21, 42, 63: ix, iy, then cx, cy
};

void free_hd_work(HdWork *w) {
    if (!w) return;
    void *ptrs[] = {w->basis, w->perm, w->et, w->eq, w->eb, w->W, w->E1, w->E2, w->ln[0], w->ln[1], w->ln[2]};
    for (void *p : ptrs)
        if (p) (void)hipFree(p);
    delete w;
}

}  // namespace swm_host

namespace {

// closure rows of both panel edges disjoint: N+1 >= 12 (sbp42), 18 (sbp63); sbp21 has one-point
// closures (any context size)
int hd_min_n(int order) { return order == 21 ? 3 : 2 * (order == 63 ? swm::Ln<63>::NB : swm::Ln<42>::NB); }

swm::HdGeo hd_geo(const swm_ctx *c) {
    swm::HdGeo g;
    const size_t P = (size_t)c->n * c->pitch;
    g.J = c->J64; g.Qi11 = c->Qi64[0]; g.Qi12 = c->Qi64[1]; g.Qi22 = c->Qi64[2];
    g.B0 = c->hd->basis; g.B1 = g.B0 + P; g.B2a = g.B0 + 2 * P; g.B2b = g.B0 + 3 * P;
    g.perm = c->hd->perm;
    g.et = c->hd->et; g.eq = c->hd->eq; g.eb = c->hd->eb;
    g.n = c->n; g.pitch = c->pitch; g.es = 4 * c->N; g.fs = c->fs; g.mps = 0;
    const double hs = c->hx * c->scale;
    g.hs2 = hs * hs;
    return g;
}

// prototype planes and the panels' signed permutations from the basis vectors b1, b2 (3 components x 6
// panels); false if a panel's components are not the prototype's
bool hd_prototype(const swm_ctx *c, const std::vector<double> &b1, const std::vector<double> &b2, std::vector<double> &basis,
                  std::vector<int> &perm) {
    const size_t n = c->n, pitch = c->pitch, P = n * pitch, last = (n - 1) * pitch + n - 1;
    auto plane = [&](const std::vector<double> &b, int k, int p) { return b.data() + (size_t)k * c->fs + p * P; };
    perm.assign(48, 0);
    basis.assign(4 * P, 0.0);
    for (int p = 0; p < 6; ++p) {
        // which component is which, from a corner, where only the prototype's zeros vanish
        int comp[3] = {-1, -1, -1};
        for (int k = 0; k < 3; ++k) comp[plane(b2, k, p)[last] == 0.0 ? 0 : plane(b1, k, p)[last] == 0.0 ? 1 : 2] = k;
        if (comp[0] < 0 || comp[1] < 0 || comp[2] < 0) return false;
        const double *src[4] = {plane(b1, comp[0], p), plane(b2, comp[1], p), plane(b1, comp[2], p), plane(b2, comp[2], p)};
        const double *zero[2] = {plane(b2, comp[0], p), plane(b1, comp[1], p)};
        const int of[4] = {0, 1, 2, 2};
        if (p == 0)
            for (int q = 0; q < 4; ++q) std::copy(src[q], src[q] + P, basis.begin() + q * P);
        double sign[3];
        for (int k = 0; k < 3; ++k) {
            sign[k] = src[k][last] * basis[k * P + last] < 0 ? -1.0 : 1.0;
            perm[8 * p + k] = comp[k];
            perm[8 * p + 4 + k] = (int)sign[k];
        }
        for (size_t j = 0; j < n; ++j) {
            int bad = 0;
            for (int q = 0; q < 4; ++q) {
                const double *x = src[q] + j * pitch, *y = basis.data() + q * P + j * pitch, s = sign[of[q]];
                for (size_t i = 0; i < n; ++i) bad |= x[i] != s * y[i];
            }
            for (const double *z : zero)
                for (size_t i = 0; i < n; ++i) bad |= z[j * pitch + i] != 0.0;
            if (bad) return false;
        }
    }
    return true;
}

// copies of every panel-edge slot (neighbour table at depth 0), its sync weights and its basis vectors
void hd_edge_tables(const swm_ctx *c, const std::vector<double> &b1, const std::vector<double> &b2, std::vector<int4> &et,
                    std::vector<double> &eq, std::vector<double> &eb) {
    const int n = c->n, es = 4 * c->N, ns = 6 * es;
    std::vector<double> qw[4];
    for (auto &v : qw) v.assign(n, 0.0);
    swmh_sync_weights(c->N, qw[0].data(), qw[1].data(), qw[2].data(), qw[3].data());
    et.resize(ns);
    eq.assign(2 * (size_t)ns, 0.0);
    eb.assign(6 * (size_t)ns, 0.0);
    auto slot = [&](int i, int j) { return j == 0 ? i : j == n - 1 ? n + i : i == 0 ? 2 * n + j - 1 : 3 * n + j - 3; };
    const size_t depths = c->host_nbr.size() / ((size_t)6 * 4 * n * 4);
    for (int p = 0; p < 6; ++p)
        for (int j = 0; j < n; ++j)
            for (int i = 0; i < n; i += j == 0 || j == n - 1 ? 1 : n - 1) {
                const int t = p * es + slot(i, j);
                int4 e = make_int4(-1, -1, 0, 0);
                for (int d = 0; d < 2; ++d) {   // 0: across an x edge, 1: across a y edge
                    const int k = d ? j : i, pos = d ? i : j;
                    if (k != 0 && k != n - 1) continue;
                    const int edge = 2 * d + (k ? 1 : 0);
                    const int *nb = &c->host_nbr[((((size_t)p * 4 + edge) * n + pos) * depths) * 4];
                    (d ? e.y : e.x) = nb[0] * es + slot(nb[1], nb[2]);
                    e.z |= nb[3] << (8 * d);
                    eq[(size_t)d * ns + t] = (d ? (k ? qw[1] : qw[0]) : (k ? qw[3] : qw[2]))[pos];
                }
                et[t] = e;
                const size_t o = ((size_t)p * n + j) * c->pitch + i;
                for (int k = 0; k < 3; ++k) {
                    eb[(size_t)k * ns + t] = b1[(size_t)k * c->fs + o];
                    eb[(size_t)(3 + k) * ns + t] = b2[(size_t)k * c->fs + o];
                }
            }
}

template <typename V>
bool hd_upload(V **dst, const std::vector<V> &src) {
    return hipMalloc((void **)dst, src.size() * sizeof(V)) == hipSuccess &&
           hipMemcpy(*dst, src.data(), src.size() * sizeof(V), hipMemcpyHostToDevice) == hipSuccess;
}

template <int ORD>
bool hd_make_weights(swm_ctx *c, double **dst) {
    using L = swm::Ln<ORD>;
    const size_t inner = (size_t)2 * (2 * L::R + 1) * c->n * c->pitch, closure = (size_t)2 * 2 * L::NB * L::NCOL * c->n;
    double *w = nullptr;
    if (hipMalloc((void **)&w, (inner + closure) * sizeof(double)) != hipSuccess) return false;
    *dst = w;
    hipLaunchKernelGGL(swm::hd_weights<ORD>, dim3((c->n * c->n + 255) / 256, 2), dim3(256), 0, nullptr, hd_geo(c), w, w + inner);
    return hipGetLastError() == hipSuccess;
}

template <int ORD>
swm::HdLn hd_ln(const swm_ctx *c) {
    using L = swm::Ln<ORD>;
    const size_t P = (size_t)c->n * c->pitch, I = (2 * L::R + 1) * P;
    const double *w = c->hd->ln[ORD == 21 ? 0 : ORD == 42 ? 1 : 2];
    return {w, w + I, w + 2 * I, w + 2 * I + (size_t)2 * L::NB * L::NCOL * c->n};
}

int ensure_hd(swm_ctx *c, int order) {
    if (c->prec != 64) return fail(SWM_EARG, "the hyperdiffusion runs in FP64 contexts only");
    if (c->n < hd_min_n(order))
        return fail(SWM_EARG, "the sbp" + std::to_string(order) + " narrow Laplacian needs N+1 >= " +
                                  std::to_string(hd_min_n(order)));
    if (!c->hd) {
        if (!c->metric_shared) return fail(SWM_EARG, "the hyperdiffusion needs the same metric on every panel");
        const size_t fb = c->field_bytes(), ns = (size_t)24 * c->N;
        std::vector<double> b1((size_t)3 * c->fs, 0.0), b2((size_t)3 * c->fs, 0.0), basis;
        std::vector<int> perm;
        swmh_basis_b(c->N, c->pitch, b1.data(), b2.data());
        if (!hd_prototype(c, b1, b2, basis, perm)) return fail(SWM_EARG, "the panels' basis vectors are not permutations of one another");
        std::vector<int4> et;
        std::vector<double> eq, eb;
        hd_edge_tables(c, b1, b2, et, eq, eb);
        HdWork *w = new HdWork();
        if (!hd_upload(&w->basis, basis) || !hd_upload(&w->perm, perm) || !hd_upload(&w->et, et) || !hd_upload(&w->eq, eq) ||
            !hd_upload(&w->eb, eb) || hipMalloc((void **)&w->W, 4 * fb) != hipSuccess ||
            hipMalloc((void **)&w->E1, 4 * ns * sizeof(double)) != hipSuccess ||
            hipMalloc((void **)&w->E2, 4 * ns * sizeof(double)) != hipSuccess ||
            hipMemset(w->W, 0, 4 * fb) != hipSuccess) {
            free_hd_work(w);
            return fail(SWM_EHIP, "hyperdiffusion work allocation failed");
        }
        c->hd = w;
        // the weights of every family that fits, here and not at its first use, which may be on another stream
        // or under capture; null-stream copies, clears and launches end before the context stream uses them
        bool ok = hd_make_weights<21>(c, &w->ln[0]);
        if (ok && c->n >= hd_min_n(42)) ok = hd_make_weights<42>(c, &w->ln[1]);
        if (ok && c->n >= hd_min_n(63)) ok = hd_make_weights<63>(c, &w->ln[2]);
        if (hipDeviceSynchronize() != hipSuccess || !ok) {
            free_hd_work(w);
            c->hd = nullptr;
            return fail(SWM_EHIP, "hyperdiffusion work allocation failed");
        }
    }
    return SWM_OK;
}

// 16 x 16 points, a thread each.  Both steps of four fields at C384 sbp42 / C191 sbp63, per pass with three
// contexts at work and in band order: 70 us / 124 us; 32 x 8 86 / 154, 16 x 8 with 128 threads 78 / 152; more threads than points, so
// that each phase of a box is one round (320 to 448), 102 to 113 / 139 to 150; two threads a point with two
// fields each 93 / 128.
constexpr int HTX = 16, HTY = 16, HSLOTS = 768;

template <int ORD, bool H, bool UV, int STEP>
int launch_lap(swm_ctx *c, const double *in, double *out, const double *Ein, double *Eout, const swm::HdFin &fin) {
    const swm::TileOrder o = swm::point_tile_order(HSLOTS, c->n, 0, c->n, swm::HdTile<ORD, HTX, HTY>::M, HTX, HTY);
    hipLaunchKernelGGL((swm::hd_lap<ORD, H, UV, STEP, HTX, HTY>), dim3(o.blocks()), dim3(HTX * HTY), 0, c->stream, o, hd_geo(c),
                       hd_ln<ORD>(c), in, out, Ein, Eout, fin);
    HIP_TRY(hipGetLastError());
    return SWM_OK;
}

// both Laplacians of the fields H / UV of a step, the second with the step's final combination
template <bool H, bool UV>
int enqueue_laps(swm_ctx *c, int order, const double *yin, const swm::HdFin &fin) {
    HdWork *w = c->hd;
    auto run = [&](auto o) {
        constexpr int ORD = decltype(o)::value;
        const int rc = launch_lap<ORD, H, UV, 1>(c, yin, w->W, nullptr, w->E1, fin);
        return rc ? rc : launch_lap<ORD, H, UV, 2>(c, w->W, nullptr, w->E1, w->E2, fin);
    };
    return order == 21 ? run(std::integral_constant<int, 21>{}) : order == 42 ? run(std::integral_constant<int, 42>{})
                                                                              : run(std::integral_constant<int, 63>{});
}

// hordiff_factory_mod.f90:25-50: the narrow-Laplacian hyperdiffusion names and their families
int hordiff_order(const char *name, const char *prefix, int &order) {
    const std::string s(name);
    for (int o : {21, 42, 63})
        if (s == prefix + std::to_string(o) + "_narrow") {
            order = o;
            return SWM_OK;
        }
    return fail(SWM_ENAME, std::string("unsupported hyperdiffusion: ") + name + " (supported: " + prefix +
                               "21_narrow, " + prefix + "42_narrow, " + prefix + "63_narrow)");
}

int parse_hordiff(const char *uv_name, const char *h_name, int &uv_order, int &h_order) {
    if (!uv_name || !h_name) return fail(SWM_EARG, "NULL hyperdiffusion name");
    int rc = hordiff_order(uv_name, "hordiff_vec_xyz_Ah_sbp_", uv_order);
    if (rc) return rc;
    return hordiff_order(h_name, "hordiff_scalar_Ah_sbp_", h_order);
}

// laplace_factory_mod.f90:20-30: the narrow-Laplacian names
int parse_laplace(const char *name, int &order) {
    if (!name) return fail(SWM_EARG, "NULL Laplacian name");
    const std::string s(name);
    if (s == "laplace_ah_sbp21_narrow") order = 21;
    else if (s == "laplace_ah_sbp42_narrow") order = 42;
    else if (s == "laplace_ah_sbp63_narrow") order = 63;
    else return fail(SWM_ENAME, "unsupported Laplacian: " + s + " (supported: laplace_ah_sbp21_narrow, "
                                    "laplace_ah_sbp42_narrow, laplace_ah_sbp63_narrow)");
    return SWM_OK;
}

// yo = y0 + dt * diff(yin) (y0 = yin = yo for the Euler step), or yo = diff(yin) with y0 = NULL
int enqueue_diff(swm_ctx *c, int uv_order, int h_order, const double *yin, const double *y0, double *yo,
                 double dt, double uv_coeff, double h_coeff) {
    // hordiff_factory_mod.f90:158-188: diff_coeff = hordiff_coeff*scale*hx, tend coefficient
    // (-1)**3 * diff_coeff**4 (the power as (c*c)*(c*c))
    const double du = uv_coeff * c->scale * c->hx, dh = h_coeff * c->scale * c->hx;
    const swm::HdFin fin{y0, yo, -1.0 * ((dh * dh) * (dh * dh)), -1.0 * ((du * du) * (du * du)), dt};
    int rc;
    // h and the velocity share the launches of one family; otherwise the velocity reads its fields before
    // any of them is written
    if (uv_order == h_order) {
        if ((rc = enqueue_laps<true, true>(c, h_order, yin, fin))) return rc;
    } else if ((rc = enqueue_laps<false, true>(c, uv_order, yin, fin)) || (rc = enqueue_laps<true, false>(c, h_order, yin, fin))) {
        return rc;
    }
    hipLaunchKernelGGL(swm::hd_edges, dim3((24 * c->N + 63) / 64), dim3(64), 0, c->stream, hd_geo(c), (const double *)c->hd->E2, fin);
    HIP_TRY(hipGetLastError());
    return SWM_OK;
}

}  // namespace

extern "C" int swm_laplace(swm_ctx *c, const char *laplace_name, const void *f, void *out) {
    if (!c || !f || !out) return fail(SWM_EARG, "NULL argument");
    if (f == out) return fail(SWM_EARG, "out must differ from f");
    int order = 0;
    int rc = parse_laplace(laplace_name, order);
    if (rc || (rc = ensure_hd(c, order))) return rc;
    const double *in = (const double *)f;
    double *res = (double *)out, *E = c->hd->E1;
    const swm::HdFin fin{};
    rc = order == 21   ? launch_lap<21, true, false, 0>(c, in, res, nullptr, E, fin)
         : order == 42 ? launch_lap<42, true, false, 0>(c, in, res, nullptr, E, fin)
                       : launch_lap<63, true, false, 0>(c, in, res, nullptr, E, fin);
    if (rc) return rc;
    hipLaunchKernelGGL(swm::hd_sync, dim3((24 * c->N + 255) / 256), dim3(256), 0, c->stream, hd_geo(c), (const double *)E, res);
    HIP_TRY(hipGetLastError());
    return SWM_OK;
}

extern "C" int swm_diff_step(swm_ctx *c, void *state, double dt, const char *hordiff_uv_name, double uv_diff_coeff,
                             const char *hordiff_h_name, double h_diff_coeff) {
    if (!c || !state) return fail(SWM_EARG, "NULL argument");
    int uv_order = 0, h_order = 0;
    int rc = parse_hordiff(hordiff_uv_name, hordiff_h_name, uv_order, h_order);
    if (rc || (rc = ensure_hd(c, uv_order)) || (rc = ensure_hd(c, h_order))) return rc;
    double *y = (double *)state;
    return enqueue_diff(c, uv_order, h_order, y, y, y, dt, uv_diff_coeff, h_diff_coeff);
}

extern "C" int swm_diff_apply(swm_ctx *c, const void *vin, void *vout, const char *hordiff_uv_name,
                              double uv_diff_coeff, const char *hordiff_h_name, double h_diff_coeff) {
    if (!c || !vin || !vout) return fail(SWM_EARG, "NULL argument");
    if (vin == vout) return fail(SWM_EARG, "vout must differ from vin");
    int uv_order = 0, h_order = 0;
    int rc = parse_hordiff(hordiff_uv_name, hordiff_h_name, uv_order, h_order);
    if (rc || (rc = ensure_hd(c, uv_order)) || (rc = ensure_hd(c, h_order))) return rc;
    return enqueue_diff(c, uv_order, h_order, (const double *)vin, nullptr, (double *)vout, 0.0, uv_diff_coeff,
                        h_diff_coeff);
}
