// The C-grid context, shared by the operators (swm_cgrid.hip) and the ECS halos (swm_cgrid_ecs.hip).
#pragma once

#include "swm_ctx.h"

namespace swmc {

constexpr int H = 4;  // halo width of the stored fields

}  // namespace swmc

struct swm_cctx {
    int N = 0, rows = 0, pitch = 0;
    long long plane = 0, fs = 0;
    double scale = 1, omega = 1, grav = 1, hx = 0;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    double *geo = nullptr;  // one panel plane each of Jo, Jx, Jy, Jq, Qi12o, Qi11x, Qi22y, Jo Qi12o, then fo (6 panels)
    double *hs = nullptr;
    // cube-edge neighbour lists (swmc::CGeo): vsrc, fsrc, osrc, qnb; signs vsg, fsg
    long long *lists = nullptr;
    signed char *signs = nullptr;
    long long *vsrc = nullptr, *fsrc = nullptr, *osrc = nullptr, *qnb = nullptr;
    signed char *vsg = nullptr, *fsg = nullptr;
    // work fields: the fluxes G (pair), the potential KE, the raw curl W, the RK accumulator and the stage
    // inputs yA, yB (a state each)
    double *work = nullptr;
    // diagnostics: quadrature weights A_centers (1..N) and A_interfaces (1..N+1) per index, block
    // partial sums (10 per block) and the 6 results
    double *qw = nullptr, *dpart = nullptr;
    long long dblocks = 0;
    StepGraphs graphs;  // captured RK4 steps of (graph_state, graph_dt)
    void *graph_state = nullptr;
    double graph_dt = 0.0;
    // ECS halos of the C grid (the vector halo and the ECS_O halo of gradient_c2_ecs and
    // massflux_c_up4), set up on first use: strip sources (normal, tangential, cells; element
    // offsets) and signs, the gathered strips, ECS_O weights, the vector tables of one (width,
    // kind) and the extended o-point array
    long long *ecs_src = nullptr;
    signed char *ecs_sign = nullptr;
    double *ecs_strips = nullptr;
    double *ecs_ow = nullptr;
    int *ecs_oind = nullptr;
    int ecs_orows = 0;
    double *ecs_vt = nullptr;
    int *ecs_vti = nullptr;
    int ecs_vt_hw = 0, ecs_vt_cov = -1;
    double *ecs_ext = nullptr;

    size_t field_bytes() const { return (size_t)fs * sizeof(double); }
    double *wf(int k) const { return work + (size_t)k * fs; }
};
