// The context behind the C ABI and what its translation units share.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/swm_gpu.h"
#include "geometry.h"
#include "swm_launch.h"

namespace swm_host {

// sets the message of swm_last_error on this thread and returns `code`
int fail(int code, const std::string &msg);

#define HIP_TRY(expr)                                                                        \
    do {                                                                                     \
        hipError_t e_ = (expr);                                                              \
        if (e_ != hipSuccess) return fail(SWM_EHIP, std::string(#expr ": ") + hipGetErrorString(e_)); \
    } while (0)

// Time steps of one state: runs of them through graphs of 4, 8, ... 64 steps, each made when a run first needs
// it; the up to three steps left over, the first run of a state, and all steps of large grids by plain
// launches.  A graph launch leaves about 10 us between two graphs where kernels follow each other in 1 to 2, so a
// graph of one step is slower than its four launches (C384 sbp42 FP64, 20 steps: 1797 us in graphs of one
// step, 1697 us by launches, 1724 us in graphs of 16 and 4).  Long graphs pay where launches cannot keep up: one
// thread driving several small grids.  Us per step by graphs / by launches, three contexts: C32 sbp42
// 9.8 / 11.7, C128 16.0 / 17.0, C256 33.8 / 34.3, C384 79.7 / 79.3; C grid C90 30.5 / 35.2, C192 60.4 / 63.1, C384
// 232.5 / 231.3; so the line lies at POINTS, between C256 and C384.  For ensembles of 64,000 to 7 million points the two are
// within 1.5 % of each other.  Making graphs costs about 7 us a step, which
// a first run of up to FIRST steps does not earn back (C90 C grid, 10 steps: 1574 us with the graphs made
// in the run, 850 us by launches).
struct StepGraphs {
    static constexpr int MIN = 4, KINDS = 5, FIRST = 128;
    static constexpr long long POINTS = 600000;
    hipGraphExec_t exec[KINDS] = {};
    bool seen = false;  // a run of the state has been made
    void drop() {
        for (hipGraphExec_t &g : exec) {
            if (g) (void)hipGraphExecDestroy(g);
            g = nullptr;
        }
        seen = false;
    }
    // nsteps of `step`, which enqueues one step of a grid of `points` points on `stream`
    template <class Step>
    int run(hipStream_t stream, long long points, int nsteps, const Step &step) {
        int rc;
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        HIP_TRY(hipStreamIsCapturing(stream, &cap));
        if (cap != hipStreamCaptureStatusNone) return fail(SWM_EHIP, "time steps cannot be captured: they run graphs of their own");
        // a first step also goes ahead of a long run: it sets up what a capture could not
        int plain = points > POINTS ? nsteps : seen ? 0 : nsteps <= FIRST ? nsteps : 1;
        for (; plain > 0; --plain, --nsteps)
            if ((rc = step())) return rc;
        seen = true;
        for (int k = KINDS - 1; k >= 0; --k) {
            const int per = MIN << k, times = nsteps / per;
            nsteps -= times * per;
            if (times && !exec[k] && (rc = make(stream, per, exec[k], step))) return rc;
            for (int q = 0; q < times; ++q) HIP_TRY(hipGraphLaunch(exec[k], stream));
        }
        for (; nsteps > 0; --nsteps)
            if ((rc = step())) return rc;
        return SWM_OK;
    }

  private:
    template <class Step>
    static int make(hipStream_t stream, int steps, hipGraphExec_t &out, const Step &step) {
        hipGraph_t g = nullptr;
        HIP_TRY(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
        int rc = SWM_OK;
        for (int q = 0; q < steps && !rc; ++q) rc = step();
        hipError_t e = hipStreamEndCapture(stream, &g);
        if (rc) { if (g) (void)hipGraphDestroy(g); return rc; }
        if (e != hipSuccess) return fail(SWM_EHIP, std::string("graph capture: ") + hipGetErrorString(e));
        e = hipGraphInstantiate(&out, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e == hipSuccess) return SWM_OK;
        out = nullptr;
        return fail(SWM_EHIP, std::string("graph instantiate: ") + hipGetErrorString(e));
    }
};

struct AdjWork;  // adjoint work space (swm_adjoint.hip), created on first use
void free_adj_work(AdjWork *w);
struct HdWork;   // hyperdiffusion work space (swm_hordiff.hip), created on first use
void free_hd_work(HdWork *w);

// one fused stage launch on the context stream (swm_capi.hip)
int run_stage(swm_ctx *c, int mode, const void *y, void *out, const void *v0, void *acc, double cy, double cacc,
              void *zeta = nullptr, const void *kin = nullptr, double ck = 0.0, double ck1 = 0.0);

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
    void *yA = nullptr, *yB = nullptr, *yC = nullptr, *curl = nullptr;
    double *red = nullptr;
    int red_blocks = 0;
    StepGraphs graphs;  // captured RK4 steps of (graph_state, graph_dt)
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
    g.hx = (T)c->hx;
    g.scale = (T)c->scale;
    g.grav = (T)c->grav;
    return g;
}

}  // namespace swm_host
