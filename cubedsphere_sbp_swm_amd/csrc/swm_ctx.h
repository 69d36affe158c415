// The context behind the C ABI and what its translation units share.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/swm_gpu.h"
#include "geometry.h"
#include "swm_launch.h"

namespace swm_host {

constexpr int RK4_GRAPH_STEPS = 50;  // steps per replay of the multi-step graph

// sets the message of swm_last_error on this thread and returns `code`
int fail(int code, const std::string &msg);

#define HIP_TRY(expr)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess) return fail(SWM_EHIP, std::string(#expr ": ") + hipGetErrorString(e_)); \
    } while (0)

struct AdjWork;  // adjoint work space (swm_adjoint.hip), created on first use
void free_adj_work(AdjWork *w);
struct HdWork;   // hyperdiffusion work space (swm_hordiff.hip), created on first use
void free_hd_work(HdWork *w);

// one fused stage launch on the context stream (swm_capi.hip)
int run_stage(swm_ctx *c, int mode, const void *y, void *out, const void *v0, void *acc, double cy, double cacc,
              void *zeta = nullptr);

}  // namespace swm_host

using namespace swm_host;

struct swm_ctx {
    int N = 0, n = 0, pitch = 0;
    long long fs = 0;
    int grad_order = 42, div_kind = 42, quad_order = 42, prec = 64;
    double scale = 1, omega = 1, grav = 1, hx = 0;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    // device geometry in the context precision
    void *J = nullptr, *Qi11 = nullptr, *Qi12 = nullptr, *Qi22 = nullptr, *f = nullptr;
    void *q[4] = {nullptr, nullptr, nullptr, nullptr};
    int4 *nbr = nullptr;
    int *einfo = nullptr;
    double *tanA = nullptr;
    bool otf = false;   // FP64: metric terms evaluated on the fly from tan(alpha)
    int tile_tx = 64, tile_ty = 8;  // tile shape of the stage kernel (swm::tile_shape_ok)
    void *hs = nullptr;
    unsigned hs_gen = 0;  // bumped whenever hs is replaced (ensemble tables hold the pointer)
    // FP64 copies used by the diagnostics
    double *J64 = nullptr, *Qi64[3] = {nullptr, nullptr, nullptr}, *f64 = nullptr, *A64 = nullptr;
    double *hs64 = nullptr;
    // RK4 work buffers (3 fields each) and diagnostics scratch
    void *yA = nullptr, *yB = nullptr, *acc = nullptr, *curl = nullptr;
    double *red = nullptr;
    int red_blocks = 0;
    // captured RK4 steps: one step, and RK4_GRAPH_STEPS steps in a row (fewer graph launches)
    hipGraphExec_t graph = nullptr, graph_multi = nullptr;
    void *graph_state = nullptr;
    double graph_dt = 0.0;
    std::vector<int> host_nbr;
    swm_host::AdjWork *adj = nullptr;
    swm_host::HdWork *hd = nullptr;
    // ECS cubic halo: weights / base indices of the last halo width used, neighbour rows
    int ecs_hw = 0;
    void *ecs_w = nullptr, *ecs_ind = nullptr, *ecs_src = nullptr;
    // ECS cubic halo on O points: weight rows set up so far, weights, base indices, edge map;
    // transform matrices of the vector halo and their rows
    int ecs_o_rows = 0, ecs_tm_rows = 0;
    void *ecs_o_w = nullptr, *ecs_o_ind = nullptr, *ecs_o_edge = nullptr, *ecs_tm = nullptr;
    // every panel holds bitwise the same J, Qi11, Qi12, Qi22 (checked at creation)
    bool metric_shared = false;

    size_t esz() const { return prec == 64 ? 8 : 4; }
    size_t field_bytes() const { return (size_t)fs * esz(); }
};

namespace swm_host {

template <typename T>
swm::DevGeo<T> make_geo(const swm_ctx *c) {
    swm::DevGeo<T> g;
    g.J = (const T *)c->J;
    g.Qi11 = (const T *)c->Qi11;
    g.Qi12 = (const T *)c->Qi12;
    g.Qi22 = (const T *)c->Qi22;
    g.f = (const T *)c->f;
    g.qb = (const T *)c->q[0];
    g.qt = (const T *)c->q[1];
    g.ql = (const T *)c->q[2];
    g.qr = (const T *)c->q[3];
    g.einfo = c->einfo;
    g.tanA = c->tanA;
    g.n = c->n;
    g.pitch = c->pitch;
    g.fs = c->fs;
    g.mps = c->metric_shared ? 0 : (long long)c->n * c->pitch;
    g.hxs = (T)(c->hx * c->scale);
    g.rhxs = T(1) / g.hxs;
    g.hx = (T)c->hx;
    g.scale = (T)c->scale;
    g.grav = (T)c->grav;
    return g;
}

}  // namespace swm_host
