// Fused RK-stage kernel of the Ah-grid vector-invariant shallow-water model (see
// swm_kernels.h for the structure) and the small kernels around it.
#include <hip/hip_runtime.h>

#include "swm_kernels.h"

namespace swm {


// LDS of one tile of TX x TY output points (one point per thread) and its halo of R points.  K lives
// on the cross-shaped region; the x-derivative inputs only on the tile rows, the y-derivative inputs
// only on the tile columns.
template <typename T, int TX, int TY, int R>
struct TileFields {
    static constexpr int LX = TX + 2 * R, LY = TY + 2 * R;
    T K[LY][LX];
    T Gxd[TY][LX], Gxc[TY][LX];
    T Gyd[LY][TX], Gyc[LY][TX];
};

// halo of a tile: what the interior rows read (tiles of interior rows only), or what any row reads
template <int ORD, bool INNER>
constexpr int tile_halo() { return INNER ? -Sbp<ORD>::INSHIFT : Sbp<ORD>::REACH; }

// LDS of one edge segment, lane l of a wave at position k0 - REACH + l along the edge: the stencil
// inputs of the own panel (side 0) and of the neighbour across the edge (side 1), and at the cube
// corners of the neighbour across the other edge (slot 0: position 0, slot 1: position n-1).
template <int ORD, typename T>
struct EdgeFields {
    static constexpr int R = Sbp<ORD>::REACH, D = Sbp<ORD>::last[0];
    T tan[2][3][64];          // depth 0: K and the two inputs of the rows along the edge
    T nrm[2][D][3][64];       // depths 0..D-1: K and the two inputs of the rows across it
    T J[2][64];
    T ctan[2][3][2 * R + 1], cnrm[2][D][3], cJ[2];
    T raw[3][4][64];          // gx, gy, div, curl before the syncs: own, neighbour, corner (lane = slot)
};

template <int ORD, typename T, int TX, int TY>
struct Smem {
    T tab[RowWeights<ORD>::SIZE];   // derivative rows (edge segments and tiles with closure rows)
    union {
        TileFields<T, TX, TY, tile_halo<ORD, true>()> in;
        TileFields<T, TX, TY, tile_halo<ORD, false>()> t;
        EdgeFields<ORD, T> e;
    };
};

// One panel edge in neighbour-table form: panel, normal axis is x, normal index of the edge
// line, tangential index = a_base + s * (local position), component code of the vector halo.
struct EdgeDesc {
    int q, nu_x, tnu, a_base, s, code;
};
__device__ __forceinline__ EdgeDesc edge_desc(const int *ei) { return {ei[0], ei[1], ei[2], ei[3], ei[4], ei[5]}; }

// Values of the output point that only the final combination reads (Coriolis parameter, RK
// stage vectors); loaded ahead of it so that their latency overlaps the stencil phases.
template <typename T>
struct OutPre {
    T f, v0[3], acc[3], kin[3];
};

template <typename T, int MODE>
__device__ __forceinline__ OutPre<T> prefetch_point(const DevGeo<T> &g, const StageArgs<T> &a, int p, unsigned off) {
    OutPre<T> o{};
    if constexpr (MODE == MODE_CURL) return o;
    const long long pb = (long long)p * g.n * g.pitch;
    o.f = at_byte(g.f + pb, off);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if constexpr (MODE == MODE_STAGE23) o.v0[k] = at_byte(a.v0 + (pb + k * g.fs), off);
        if constexpr (MODE == MODE_SLOPE3) {
            o.v0[k] = at_byte(a.y + (pb + k * g.fs), off);
            o.kin[k] = at_byte(a.kin + (pb + k * g.fs), off);
        }
        if constexpr (MODE == MODE_STAGE23 || MODE == MODE_STAGE4 || MODE == MODE_SLOPE3) o.acc[k] = at_byte((const T *)a.acc + (pb + k * g.fs), off);
    }
    return o;
}

// Coriolis term, tendencies and RK stage combination of one point
// (coriolis_colocated_mod.f90:97-98, operator_swm_mod.f90:95-101, rk4_mod.f90:28-40)
// hu = h*ut, hv = h*vt: the mass fluxes of the point (u, v are read by stage 1 only)
template <typename T, int MODE>
__device__ __forceinline__ void finish_point(const DevGeo<T> &g, const StageArgs<T> &a, int p, unsigned off, T h, T u,
                                             T v, T hu, T hv, T Jv, T gx, T gy, T dv, T cu, const OutPre<T> &pre) {
    const long long pb = (long long)p * g.n * g.pitch;
    T *out = a.out + pb;
    if constexpr (MODE == MODE_CURL) {
        at_byte(out, off) = cu;
        return;
    }
    if (a.zeta) at_byte(a.zeta + pb, off) = cu;
    const T fz = pre.f + cu;
    const T cor_u = fz * hv / h * Jv;
    const T cor_v = -(fz * hu / h * Jv);
    const T k[3] = {-dv, -gx + cor_u, -gy + cor_v}, y[3] = {h, u, v};
    T *acc = a.acc + pb;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const long long fc = c * g.fs;
        if constexpr (MODE == MODE_RHS || MODE == MODE_SLOPE2) {
            at_byte(out + fc, off) = k[c];
        } else if constexpr (MODE == MODE_STAGE1) {
            at_byte(out + fc, off) = y[c] + a.cy * k[c];
            at_byte(acc + fc, off) = y[c] + a.cacc * k[c];
        } else if constexpr (MODE == MODE_STAGE23) {
            at_byte(out + fc, off) = pre.v0[c] + a.cy * k[c];
            at_byte(acc + fc, off) = pre.acc[c] + a.cacc * k[c];
        } else if constexpr (MODE == MODE_SLOPE3) {
            at_byte(out + fc, off) = pre.v0[c] + a.cy * k[c];
            at_byte(acc + fc, off) = ((pre.v0[c] + a.ck1 * pre.acc[c]) + a.cacc * pre.kin[c]) + a.cacc * k[c];
        } else if constexpr (MODE == MODE_STAGE4) {
            at_byte(out + fc, off) = pre.acc[c] + a.cy * k[c];
        }
    }
}

// the derivative rows from memory into LDS; the caller's barrier follows
template <int ORD, typename T>
__device__ __forceinline__ void load_rows(T *tab, int tid, int nthreads) {
    for (int c = tid; c < RowWeights<ORD>::SIZE; c += nthreads) tab[c] = (T)row_weights<ORD>.w[c];
}

// One TX x TY tile of panel p starting at (tx0, ty0) >= (1, 1): the whole RHS + RK stage update
// of its points off the panel edges (the panel-edge points belong to the edge segments).
// INNER (inner_tile): every derivative row of the tile is an interior one, so every point of it and
// of its halo exists and none is on a panel edge; its halo is the REACH of the interior row (2 points
// for sbp42 and sbp43, 3 for sbp63, against 3, 5, 5 for the closure rows), its guards vanish and its
// rows have constant weights.  The other tiles take their rows from the table.
// At C384 sbp42 FP64 (64 x 8, metric read) an RK4 step takes 83 us by slopes and 85 us by states, 21.3 us per
// stage: a stage 2/3 by states moves about 135 MB at nearly the 7 TB/s that a copy of cache-resident buffers of
// this size reaches.  With three contexts at work the states no longer fit the memory-side cache: 80 us by slopes, 91 by
// states.  Wider halos, a branch and its code per closure row, 64-bit offsets and panel-major tile order (metric
// read once per panel) took 24-25 us a stage.
template <int ORD, typename T, int MODE, int TX, int TY, bool OTF, bool PERSIST, bool INNER>
__device__ __forceinline__ void stage_tile(const DevGeo<T> &g, const StageArgs<T> &a, int p, int tx0, int ty0,
                                           TileFields<T, TX, TY, tile_halo<ORD, INNER>()> &sm, T *tab) {
    constexpr int R = tile_halo<ORD, INNER>(), NT = TX * TY;
    const int n = g.n;
    // in the persistent ensemble loop the thread index is made opaque per tile, so that the
    // thread-index arithmetic is recomputed per tile instead of being hoisted out of the loop
    // and held in registers
    int tid = threadIdx.x;
    if constexpr (PERSIST) asm volatile("" : "+v"(tid));
    const PanelIn<T> in = panel_in(g, a, p);

    // ---- load phase: every thread loads its own tile point (kept in registers for the output
    // phase), plus at most NH halo points, the y-halo rows first (whole waves), then the x-halo
    // columns; all global loads are issued before any derived value is formed, so that they are in
    // flight together. ----
    constexpr int NYH = 2 * R * TX, NXH = 2 * R * TY, NH = (NYH + NXH + NT - 1) / NT;
    const int tx = tid % TX, ty = tid / TX;
    const int i = tx0 + tx, j = ty0 + ty;
    const bool own_ok = INNER || (i < n && j < n);
    RawPoint<T> own{};
    if (own_ok) own = load_point<MODE, OTF>(g, in, i, j);
    RawPoint<T> rh[NH];
    int hc[NH], hr[NH];   // tile column and row of the halo point, relative to (tx0, ty0)
    bool okh[NH];
#pragma unroll
    for (int k = 0; k < NH; ++k) {
        const int c = tid + k * NT;
        if (c < NYH) {
            const int r = c / TX;
            hc[k] = c - r * TX;
            hr[k] = r < R ? r - R : r - R + TY;
        } else {
            const int q = c - NYH, r = q / (2 * R), x = q - r * (2 * R);
            hr[k] = r;
            hc[k] = x < R ? x - R : x - R + TX;
        }
        okh[k] = c < NYH + NXH;
        if constexpr (!INNER) {
            const int hi = tx0 + hc[k], hj = ty0 + hr[k];
            okh[k] = okh[k] && hi >= 0 && hj >= 0 && hi < n && hj < n;
        }
        if (okh[k]) rh[k] = load_point<MODE, OTF>(g, in, tx0 + hc[k], ty0 + hr[k]);
    }
    if constexpr (!INNER) load_rows<ORD, T>(tab, tid, NT);
    // of the own point only h, u, v, J and the mass fluxes h*ut, h*vt stay live for the output
    // phase (the same products the Coriolis term forms)
    T own_hu = T(0), own_hv = T(0);
    if (own_ok) {
        const Derived<T> d = derived_of<MODE>(g, own, in.ck);
        own_hu = d.hu;
        own_hv = d.hv;
        sm.K[ty + R][tx + R] = d.K;
        sm.Gxd[ty][tx + R] = d.Gxd;
        sm.Gxc[ty][tx + R] = d.Gxc;
        sm.Gyd[ty + R][tx] = d.Gyd;
        sm.Gyc[ty + R][tx] = d.Gyc;
    }
#pragma unroll
    for (int k = 0; k < NH; ++k) {
        if (!okh[k]) continue;
        const Derived<T> d = derived_of<MODE>(g, rh[k], in.ck);
        sm.K[hr[k] + R][hc[k] + R] = d.K;
        if (tid + k * NT < NYH) {
            sm.Gyd[hr[k] + R][hc[k]] = d.Gyd;
            sm.Gyc[hr[k] + R][hc[k]] = d.Gyc;
        } else {
            sm.Gxd[hr[k]][hc[k] + R] = d.Gxd;
            sm.Gxc[hr[k]][hc[k] + R] = d.Gxc;
        }
    }
    // the output point's Coriolis parameter and RK vectors: issued after the load phase (issued
    // with it, they raised its register peak by 14 VGPRs at FP64), in flight across the barrier and
    // the stencil phase
    const bool out_ok = INNER || (i < n - 1 && j < n - 1);
    const unsigned off = point_off(g, i, j);
    OutPre<T> pre{};
    if (out_ok) pre = prefetch_point<T, MODE>(g, a, p, off);
    __syncthreads();

    // ---- output phase: the thread's own point ----
    if (!out_ok) return;
    const int lx = tx + R, ly = ty + R;
    T dxK, dyK, dxD, dyD, dxC, dyC;
    if constexpr (INNER) {
        dxK = sbp_row_in<ORD, T>(lx, [&](int q) { return sm.K[ly][q]; });
        dyK = sbp_row_in<ORD, T>(ly, [&](int q) { return sm.K[q][lx]; });
        dxD = sbp_row_in<ORD, T>(lx, [&](int q) { return sm.Gxd[ty][q]; });
        dyD = sbp_row_in<ORD, T>(ly, [&](int q) { return sm.Gyd[q][tx]; });
        dxC = sbp_row_in<ORD, T>(lx, [&](int q) { return sm.Gxc[ty][q]; });
        dyC = sbp_row_in<ORD, T>(ly, [&](int q) { return sm.Gyc[q][tx]; });
    } else {
        const RowAt rx = row_at<ORD>(i, n), ry = row_at<ORD>(j, n);
        const int bx = rx.base - tx0 + R, by = ry.base - ty0 + R;
        row_apply3<ORD, T>(tab, rx, [&](int m, T &x, T &y, T &z) {
            x = sm.K[ly][bx + m]; y = sm.Gxd[ty][bx + m]; z = sm.Gxc[ty][bx + m];
        }, dxK, dxD, dxC);
        row_apply3<ORD, T>(tab, ry, [&](int m, T &x, T &y, T &z) {
            x = sm.K[by + m][lx]; y = sm.Gyd[by + m][tx]; z = sm.Gyc[by + m][tx];
        }, dyK, dyD, dyC);
    }
    const T Jd = own.J * g.hx * g.scale;
    finish_point<T, MODE>(g, a, p, off, own.h, own.u, own.v, own_hu, own_hv, own.J, dxK / g.hxs, dyK / g.hxs,
                          (dxD + dyD) / Jd, (dxC + dyC) / Jd, pre);
}

// Edge segment `seg` of the cube (edge_segs(n, REACH) per cube): positions k0..k1-1 of one panel
// edge, at most 64 - 2 REACH points.  Both panels' stencil inputs along the edge go to LDS, one line of
// one depth per wave; then one wave per panel forms the raw values of its side's one-sided rows (a
// third those of the corners' third panel), and the first wave applies the scalar and covariant
// vector edge syncs (ecs_Ah_vec_sync_mod.f90:77-124 with (U, V) = (gy, gx),
// halo_Ah_scalar_sync_mod.f90:52-93, in the reference's operand order) and the RK stage update.
// These blocks are the longest chains of a launch on small panels, and most of such a chain is
// fetching its instructions, which no earlier wave has brought in: every phase therefore has one
// copy of its code, for all depths, sides and closure rows.  The kernel is 14 KB (sbp42) / 17 KB (sbp63)
// instead of 71 / 147 KB with the rows written out per side; a C95 sbp63 step went from 34 to 19 us and the
// 16-member ensemble (C48-C192) from 342 to 239 us.
template <int ORD, typename T, int MODE, bool OTF, bool PERSIST = false>
__device__ __forceinline__ void stage_edge(const DevGeo<T> &g, const StageArgs<T> &a, int seg, EdgeFields<ORD, T> &sm,
                                           T *tab, int nthreads) {
    constexpr int R = Sbp<ORD>::REACH, D = Sbp<ORD>::last[0], S = edge_seg_len(R);
    constexpr int NE = Sbp<ORD>::NE;
    const int n = g.n;
    int tid = threadIdx.x;
    if constexpr (PERSIST) asm volatile("" : "+v"(tid));
    const int nsx = edge_segs_x(n, R), nsy = edge_segs_y(n, R), per = 2 * (nsx + nsy);
    const int p = seg / per, r = seg - p * per;
    int e, si;
    if (r < 2 * nsx) { e = r / nsx; si = r - e * nsx; }
    else { e = 2 + (r - 2 * nsx) / nsy; si = r - 2 * nsx - (e - 2) * nsy; }
    const int k0 = e < 2 ? si * S : 1 + si * S;
    const int k1 = e < 2 ? min(n, k0 + S) : min(n - 1, k0 + S);
    // side 0: the own panel in neighbour-table form (identity orientation); side 1: across e
    const EdgeDesc own{p, e < 2 ? 1 : 0, (e == 0 || e == 2) ? 0 : n - 1, 0, 1, 0};
    const EdgeDesc nbr = edge_desc(g.einfo + (p * 4 + e) * 8);
    // cube corners of the x-edges: the neighbour across the y-edge at i = 0 / n-1
    const bool c0 = e < 2 && k0 == 0, c1 = e < 2 && k1 == n;
    const int ci = e == 0 ? 0 : n - 1;

    const int lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), nwaves = nthreads / 64;
    const int k = k0 - R + lane;
    const bool act = k >= k0 && k < k1;
    const int i = e < 2 ? ci : k, j = e < 2 ? k : (e == 2 ? 0 : n - 1);
    const unsigned off = point_off(g, i, j);
    OutPre<T> pre{};
    T q = T(0);          // sync weight of the own point; at a corner the x-edge's, qc the y-edge's
    T qc = T(0);
    if (wave == 0 && act) {
        pre = prefetch_point<T, MODE>(g, a, p, off);
        q = e == 0 ? g.ql[k] : e == 1 ? g.qr[k] : e == 2 ? g.qb[k] : g.qt[k];
        if (e < 2 && k == 0) qc = g.qb[i];
        if (e < 2 && k == n - 1) qc = g.qt[i];
    }

    // ---- inputs: line w of the list (side 0 depths 0..D-1, side 1 likewise, corner slots 0, 1) ----
    RawPoint<T> mine{};
    T hu = T(0), hv = T(0);
#pragma unroll 1
    for (int w = wave; w < 2 * D + 2; w += nwaves) {
        const bool corner = w >= 2 * D;
        const int side = corner ? w - 2 * D : (w >= D ? 1 : 0);   // or corner slot
        EdgeDesc ei = side ? nbr : own;
        int d = w - side * D, kk = k;
        bool ok = kk >= 0 && kk < n && (d == 0 || act);
        if (corner) {
            if (!(side == 0 ? c0 : c1)) continue;
            ei = edge_desc(g.einfo + (p * 4 + 2 + side) * 8);
            d = lane <= 2 * R ? 0 : lane - 2 * R;
            kk = lane <= 2 * R ? ci - R + lane : ci;
            ok = kk >= 0 && kk < n && d < D;
        }
        if (!ok) continue;
        const int nidx = ei.tnu == 0 ? d : n - 1 - d, tidx = ei.a_base + ei.s * kk;
        const PanelIn<T> in = panel_in(g, a, ei.q);
        RawPoint<T> rp = load_point<MODE, OTF>(g, in, ei.nu_x ? nidx : tidx, ei.nu_x ? tidx : nidx);
        const Derived<T> dv = derived_of<MODE>(g, rp, in.ck);
        const T nD = ei.nu_x ? dv.Gxd : dv.Gyd, nC = ei.nu_x ? dv.Gxc : dv.Gyc;
        const T tD = ei.nu_x ? dv.Gyd : dv.Gxd, tC = ei.nu_x ? dv.Gyc : dv.Gxc;
        if (!corner) {
            sm.nrm[side][d][0][lane] = dv.K;
            sm.nrm[side][d][1][lane] = nD;
            sm.nrm[side][d][2][lane] = nC;
            if (d == 0) {
                sm.tan[side][0][lane] = dv.K;
                sm.tan[side][1][lane] = tD;
                sm.tan[side][2][lane] = tC;
                sm.J[side][lane] = rp.J;
            }
            if (w == 0) {      // the first wave's first line: its lanes' output points
                mine = rp;
                hu = dv.hu;
                hv = dv.hv;
            }
        } else {
            if (kk == ci) {
                sm.cnrm[side][d][0] = dv.K;
                sm.cnrm[side][d][1] = nD;
                sm.cnrm[side][d][2] = nC;
                if (d == 0) sm.cJ[side] = rp.J;
            }
            if (d == 0) {
                sm.ctan[side][0][lane] = dv.K;
                sm.ctan[side][1][lane] = tD;
                sm.ctan[side][2][lane] = tC;
            }
        }
    }
    load_rows<ORD, T>(tab, tid, nthreads);
    __syncthreads();

    // ---- raw values: wave 0 the own panel's, wave 1 the neighbour's, wave 2 lanes 0, 1 the corners' ----
    if (wave < 2 ? act : (wave == 2 && lane < 2 && (lane == 0 ? c0 : c1))) {
        const bool corner = wave == 2;
        EdgeDesc ed = wave ? nbr : own;
        int kk = k, ns = 64, ts = 64;
        const T *nb = &sm.nrm[wave & 1][0][0][lane], *tb = &sm.tan[wave & 1][0][lane], *Jb = &sm.J[wave & 1][lane];
        if (corner) {
            ed = edge_desc(g.einfo + (p * 4 + 2 + lane) * 8);
            kk = ci;
            ns = 1;
            ts = 2 * R + 1;
            nb = sm.cnrm[lane][0];
            tb = &sm.ctan[lane][0][R];
            Jb = &sm.cJ[lane];
        }
        // across the edge: row 0 by depth, or the last row, whose inputs run from depth D-1 to 0
        const bool low = ed.tnu == 0;
        T nK, nD, nC, tK, tD, tC;
        row_apply3<ORD, T>(tab, RowAt{0, D, low ? 0 : 2 * NE}, [&](int m, T &x, T &y, T &z) {
            const T *q = nb + (low ? m : D - 1 - m) * 3 * ns;
            x = q[0]; y = q[ns]; z = q[2 * ns];
        }, nK, nD, nC);
        // along it: index b of the panel lies s (b - a0) lanes away
        const int a0 = ed.a_base + ed.s * kk;
        const RowAt rt = row_at<ORD>(a0, n);
        row_apply3<ORD, T>(tab, rt, [&](int m, T &x, T &y, T &z) {
            const T *q = tb + ed.s * (rt.base + m - a0);
            x = q[0]; y = q[ts]; z = q[2 * ts];
        }, tK, tD, tC);
        const T Jd = *Jb * g.hx * g.scale;
        // x before y in the sums: the operands commute, so the order does not matter
        sm.raw[wave][0][lane] = (ed.nu_x ? nK : tK) / g.hxs;
        sm.raw[wave][1][lane] = (ed.nu_x ? tK : nK) / g.hxs;
        sm.raw[wave][2][lane] = (nD + tD) / Jd;
        sm.raw[wave][3][lane] = (nC + tC) / Jd;
    }
    __syncthreads();
    if (wave != 0 || !act) return;

    T gx = sm.raw[0][0][lane], gy = sm.raw[0][1][lane], dv = sm.raw[0][2][lane], cu = sm.raw[0][3][lane];
    const T U = gy, V = gx;
    // the neighbour's raw values mapped to this panel's components (vector halo convention)
    T Vn, Un;
    map_vec(nbr.code, sm.raw[1][0][lane], sm.raw[1][1][lane], Vn, Un);
    const T Dn = sm.raw[1][2][lane], Cn = sm.raw[1][3][lane];
    if (e < 2 && (k == 0 || k == n - 1)) {
        const int slot = k == 0 ? 0 : 1;
        T Vy, Uy;
        map_vec(g.einfo[(p * 4 + 2 + slot) * 8 + 5], sm.raw[2][0][slot], sm.raw[2][1][slot], Vy, Uy);
        dv = (dv + Dn + sm.raw[2][2][slot]) / T(3);
        cu = (cu + Cn + sm.raw[2][3][slot]) / T(3);
        gy = (U + Un + Uy + qc * Vy) / T(3);
        gx = (V + Vn + Vy + q * Un) / T(3);
    } else {
        // the component along the edge is averaged, the one across it takes the weight q
        dv = T(0.5) * (dv + Dn);
        cu = T(0.5) * (cu + Cn);
        if (e < 2) {
            gy = T(0.5) * (U + Un);
            gx = T(0.5) * (V + Vn + q * Un);
        } else {
            gx = T(0.5) * (V + Vn);
            gy = T(0.5) * (U + Un + q * Vn);
        }
    }
    finish_point<T, MODE>(g, a, p, off, mine.h, mine.u, mine.v, hu, hv, mine.J, gx, gy, dv, cu, pre);
}

// a tile starting at (tx0, ty0) whose derivative rows are all interior ones (NE <= i, j < n - NE; the
// interior row's reach is at most NE, so its halo lies inside the panel)
template <int ORD, int TX, int TY>
__device__ __forceinline__ bool inner_tile(int tx0, int ty0, int n) {
    constexpr int NE = Sbp<ORD>::NE;
    static_assert(tile_halo<ORD, true>() <= NE, "the halo of an inner tile lies inside the panel");
    return tx0 >= NE && tx0 + TX <= n - NE && ty0 >= NE && ty0 + TY <= n - NE;
}

// Tile t of a cube: row strips outermost, then panels, then the columns of a strip.  An XCD's
// contiguous range (xcd_tile) is then a band of rows of all six panels, which read the same metric
// planes there: an eighth of them per XCD, which stays in its L2 from panel to panel.
template <int ORD, typename T, int MODE, int TX, int TY, bool OTF, bool PERSIST>
__device__ __forceinline__ void stage_any_tile(const DevGeo<T> &g, const StageArgs<T> &a, int t,
                                               Smem<ORD, T, TX, TY> &sm) {
    const int ntx = tiles_along(g.n, TX);
    const int strip = t / (6 * ntx), rem = t - strip * 6 * ntx, p = rem / ntx;
    const int tx0 = 1 + (rem - p * ntx) * TX, ty0 = 1 + strip * TY;
    if (inner_tile<ORD, TX, TY>(tx0, ty0, g.n))
        stage_tile<ORD, T, MODE, TX, TY, OTF, PERSIST, true>(g, a, p, tx0, ty0, sm.in, sm.tab);
    else
        stage_tile<ORD, T, MODE, TX, TY, OTF, PERSIST, false>(g, a, p, tx0, ty0, sm.t, sm.tab);
}

// edge blocks first (a multiple of 8, so that the tiles keep their XCD-contiguous mapping)
SWM_HD constexpr int edge_blocks(int n, int reach) { return (edge_segs(n, reach) + 7) / 8 * 8; }

template <int ORD, typename T, int MODE, int TX, int TY, bool OTF>
__global__ void __launch_bounds__(TX * TY) stage_kernel(DevGeo<T> g, StageArgs<T> a) {
    __shared__ Smem<ORD, T, TX, TY> sm;
    const int ne = edge_blocks(g.n, Sbp<ORD>::REACH);
    if ((int)blockIdx.x < ne) {
        if ((int)blockIdx.x < edge_segs(g.n, Sbp<ORD>::REACH))
            stage_edge<ORD, T, MODE, OTF>(g, a, blockIdx.x, sm.e, sm.tab, TX * TY);
        return;
    }
    const int ntiles = 6 * tiles_along(g.n, TX) * tiles_along(g.n, TY);
    stage_any_tile<ORD, T, MODE, TX, TY, OTF, false>(g, a, xcd_tile(blockIdx.x - ne, ntiles), sm);
}

// Copy of a block-uniform struct into scalar registers (word by word through readfirstlane):
// the stores of the stage body keep the compiler from proving the table unchanged, which it
// would need to use scalar loads by itself.
template <typename S>
__device__ __forceinline__ S uniform_copy(const S *src) {
    static_assert(sizeof(S) % 4 == 0, "word-sized struct");
    S out;
    const unsigned *w = reinterpret_cast<const unsigned *>(src);
    unsigned *o = reinterpret_cast<unsigned *>(&out);
#pragma unroll
    for (int k = 0; k < (int)(sizeof(S) / 4); ++k) o[k] = __builtin_amdgcn_readfirstlane(w[k]);
    return out;
}

// Ensemble of cubes of different sizes in one launch: the blocks walk the concatenated task list
// of all members (per member its 6*ntx*nty tiles (tiles_along), then its edge_segs(n, REACH) edge
// segments), XCD-contiguous; a persistent grid loops over it, a grid of one block per task runs
// each block once.  tasks[t] = (member, task index within the
// member): one load gives a block its member, whose geometry and stage arguments it then takes
// from the member table.
template <int ORD, typename T, int MODE, int TX, int TY, bool OTF>
__global__ void __launch_bounds__(TX * TY) ens_stage_kernel(const EnsMember<T> *__restrict__ members,
                                                            const int2 *__restrict__ tasks, int ntiles) {
    __shared__ Smem<ORD, T, TX, TY> sm;
    for (int it = blockIdx.x; it < ntiles; it += gridDim.x) {
        const int tile = xcd_tile(it, ntiles);
        const int2 tk = tasks[tile];
        const int m = __builtin_amdgcn_readfirstlane(tk.x);   // block-uniform member index
        const int lt = __builtin_amdgcn_readfirstlane(tk.y);
        const DevGeo<T> g = uniform_copy(&members[m].g);
        const StageArgs<T> a = uniform_copy(&members[m].a);
        const int ncell = 6 * tiles_along(g.n, TX) * tiles_along(g.n, TY);
        __syncthreads();  // the previous task's LDS reads are done
        if (lt >= ncell)
            stage_edge<ORD, T, MODE, OTF, true>(g, a, lt - ncell, sm.e, sm.tab, TX * TY);
        else
            stage_any_tile<ORD, T, MODE, TX, TY, OTF, true>(g, a, lt, sm);
    }
}

}  // namespace swm

namespace swm {

template <int ORD, typename T, int TX, int TY, bool OTF>
hipError_t launch_one(int mode, const DevGeo<T> &g, const StageArgs<T> &a, hipStream_t s) {
    const int ntx = tiles_along(g.n, TX), nty = tiles_along(g.n, TY);
    const dim3 grid(edge_blocks(g.n, Sbp<ORD>::REACH) + 6 * ntx * nty), block(TX * TY);
    switch (mode) {
    case MODE_RHS: hipLaunchKernelGGL((stage_kernel<ORD, T, MODE_RHS, TX, TY, OTF>), grid, block, 0, s, g, a); break;
    case MODE_STAGE1: hipLaunchKernelGGL((stage_kernel<ORD, T, MODE_STAGE1, TX, TY, OTF>), grid, block, 0, s, g, a); break;
    case MODE_STAGE23: hipLaunchKernelGGL((stage_kernel<ORD, T, MODE_STAGE23, TX, TY, OTF>), grid, block, 0, s, g, a); break;
    case MODE_STAGE4: hipLaunchKernelGGL((stage_kernel<ORD, T, MODE_STAGE4, TX, TY, OTF>), grid, block, 0, s, g, a); break;
    case MODE_SLOPE2: hipLaunchKernelGGL((stage_kernel<ORD, T, MODE_SLOPE2, TX, TY, OTF>), grid, block, 0, s, g, a); break;
    case MODE_SLOPE3: hipLaunchKernelGGL((stage_kernel<ORD, T, MODE_SLOPE3, TX, TY, OTF>), grid, block, 0, s, g, a); break;
    case MODE_CURL: hipLaunchKernelGGL((stage_kernel<ORD, T, MODE_CURL, TX, TY, OTF>), grid, block, 0, s, g, a); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int ORD, typename T, int TX, int TY, bool OTF, int MODE>
hipError_t launch_ens_mode(const EnsLaunch &r) {
    auto kern = ens_stage_kernel<ORD, T, MODE, TX, TY, OTF>;
    static int per_cu = 0;  // resident blocks per CU of this instantiation
    if (per_cu == 0) {
        int nb = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kern, TX * TY, 0);
        if (e != hipSuccess) return e;
        per_cu = nb > 0 ? nb : 1;
    }
    // resident blocks x the requested waves of blocks (0: one block per task); a multiple of 8
    // keeps a block's tiles on its XCD
    long long grid = r.blocks_per_slot > 0 ? (long long)r.num_cu * per_cu * r.blocks_per_slot : (long long)r.ntiles;
    grid = (grid + 7) / 8 * 8;
    if (grid > r.ntiles) grid = (r.ntiles + 7) / 8 * 8;
    if (grid < 8) grid = 8;
    hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(TX * TY), 0, r.stream, (const EnsMember<T> *)r.members,
                       r.tasks, r.ntiles);
    return hipGetLastError();
}

template <int ORD, typename T, int TX, int TY, bool OTF>
hipError_t launch_ens_one(const EnsLaunch &r) {
    switch (r.mode) {
    case MODE_STAGE1: return launch_ens_mode<ORD, T, TX, TY, OTF, MODE_STAGE1>(r);
    case MODE_STAGE23: return launch_ens_mode<ORD, T, TX, TY, OTF, MODE_STAGE23>(r);
    case MODE_STAGE4: return launch_ens_mode<ORD, T, TX, TY, OTF, MODE_STAGE4>(r);
    default: return hipErrorInvalidValue;
    }
}

// the tile shapes of the stage kernels (tile_shape_ok): 64 x 8, 32 x 16, 16 x 32 (512 threads)
// and 32 x 8 (256 threads)
template <int ORD, typename T, bool OTF>
hipError_t launch_ens_shape(const EnsLaunch &r) {
    if (r.tx == 64 && r.ty == 8) return launch_ens_one<ORD, T, 64, 8, OTF>(r);
    if (r.tx == 32 && r.ty == 16) return launch_ens_one<ORD, T, 32, 16, OTF>(r);
    if (r.tx == 16 && r.ty == 32) return launch_ens_one<ORD, T, 16, 32, OTF>(r);
    if (r.tx == 32 && r.ty == 8) return launch_ens_one<ORD, T, 32, 8, OTF>(r);
    return hipErrorInvalidValue;
}

template <int ORD>
hipError_t launch_ens_f64(const EnsLaunch &r) {
    return r.otf ? launch_ens_shape<ORD, double, true>(r) : launch_ens_shape<ORD, double, false>(r);
}

template <int ORD>
hipError_t launch_ens_f32(const EnsLaunch &r) {
    return launch_ens_shape<ORD, float, false>(r);
}

template <int ORD, typename T, bool OTF>
hipError_t launch_stage_shape(const StageLaunch &r, const DevGeo<T> &g, const StageArgs<T> &a) {
    if (r.tx == 64 && r.ty == 8) return launch_one<ORD, T, 64, 8, OTF>(r.mode, g, a, r.stream);
    if (r.tx == 32 && r.ty == 16) return launch_one<ORD, T, 32, 16, OTF>(r.mode, g, a, r.stream);
    if (r.tx == 16 && r.ty == 32) return launch_one<ORD, T, 16, 32, OTF>(r.mode, g, a, r.stream);
    if (r.tx == 32 && r.ty == 8) return launch_one<ORD, T, 32, 8, OTF>(r.mode, g, a, r.stream);
    return hipErrorInvalidValue;
}

template <int ORD>
hipError_t launch_stage_f64(const StageLaunch &r) {
    return r.otf ? launch_stage_shape<ORD, double, true>(r, r.gd, r.ad) : launch_stage_shape<ORD, double, false>(r, r.gd, r.ad);
}

template <int ORD>
hipError_t launch_stage_f32(const StageLaunch &r) {
    return launch_stage_shape<ORD, float, false>(r, r.gf, r.af);
}

}  // namespace swm
