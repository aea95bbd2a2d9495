// bgf_capi.cpp -- extern "C" entry points of libbgflood_amd.so (declared in
// include/bgflood_amd.h).  A handle owns the device Model<T> of one domain:
// the state in two buffers (evolv and evolv_o of src/Arrays.h:300-354, used
// as a ping-pong pair), the static bed and friction arrays, the predictor
// tendencies (Model.adv), the block description and a device-resident loop
// state.  Between API calls the current state is always in buffer 0
// (evolv).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/bgflood_amd.h"
#include "bgf_host.h"

using namespace bgf_host;

// A boundary segment as set: type, the side whose strip it is (0..3) or its
// polygon (side -1), its level series, and its level map (device frames and
// the map of the current step, or the caller's device map read in place).
struct HostSeg {
    int type = 1, side = -1;
    Polygon poly;
    std::vector<double> t, z;
    double* d_series = nullptr;  // t, then z
    float* d_frames = nullptr;
    float* d_now = nullptr;
    const float* ext_now = nullptr;
    int nx = 0, ny = 0, nt = 0;
    double xo = 0, yo = 0, dx = 0, dy = 0, to = 0, tdt = 0;
};

inline void free_seg(HostSeg& g) {
    if (g.d_series) (void)hipFree(g.d_series);
    if (g.d_frames) (void)hipFree(g.d_frames);
    if (g.d_now) (void)hipFree(g.d_now);
    g.d_series = nullptr;
    g.d_frames = g.d_now = nullptr;
}

struct bgf_handle_s {
    bgf_param p;
    int prec;
    size_t es;  // element size
    int nblk, nblkmem;
    size_t S;   // elements per array
    std::vector<int> active;
    // one allocation that holds the mesh's arrays and the loop state, and on multi-level meshes the
    // cells' arrays and the staging of bgf_remesh as well (device_room)
    void* arena = nullptr;
    int *d_active = nullptr, *d_order = nullptr, *d_level = nullptr;
    int* d_queue = nullptr;  // work-queue counters of the persistent kernels
    int* d_rec = nullptr;    // per-position block records of the processing order
    bool cf_shared = false;  // the caller holds the cf device array
    int *d_nb[8] = {nullptr};  // LeftBot LeftTop RightBot RightTop TopLeft TopRight BotLeft BotRight
    int* d_nbr = nullptr;      // multi-level meshes: the neighbour record of each block slot (bgf::NBR ints)
    int4* d_rcell = nullptr;   // their gather recipes (bgf::RECIPES per slot)
    int2* d_rmeta = nullptr;
    int* d_fix = nullptr;      // and the blocks whose advance waits for other blocks' faces
    void *d_h[2] = {nullptr, nullptr}, *d_u[2] = {nullptr, nullptr}, *d_v[2] = {nullptr, nullptr};
    void *d_zb = nullptr, *d_cf = nullptr, *d_dh = nullptr, *d_dhu = nullptr, *d_dhv = nullptr;
    double *d_volpart = nullptr, *d_volout = nullptr;
    bgf::DevLoop* d_loop = nullptr;  // two loop states: a step takes one and leaves the next in the other
    int loop_at = 0;                 // the one that the enqueued work leaves last
    bgf::KParams kp;
    hipStream_t stream = nullptr;
    std::unique_ptr<ReadBack> back{new ReadBack};
    bool timing = false;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    double t_pred = 0, t_red = 0, t_corr = 0;
    int t_n = 0;
    int pending_steps = 0;  // steps enqueued by bgf_run_async
    bool state_set = false;
    bgf::LoopState* loop_host = nullptr;  // pinned: the loop state after the enqueued work
    // output statistics (Calcmeanmax): enabled set, arrays, steps since the means were reset
    bgf::StatsLaunch stats{};
    int stats_n = 0;
    // multi-level meshes: the step runs the bgf_amr kernels on the reference
    // layout (state stays in buffer 0, buffer 1 is evolv_o)
    bool amr = false;
    int* d_inv = nullptr;
    void* d_amr[11] = {nullptr};  // 0-1: remesh staging of the bed and roughness; 2-9: face fluxes; 10: hsnap
    void* d_ch = nullptr;          // compensation of h (BGF_FP32_COMP)
    void* d_metric = nullptr;      // spherical metric terms per block
    bool use_graph = true;
    hipGraphExec_t graph = nullptr;  // PERIOD steps, captured on first use
    int last_steps = 0;              // steps taken by the last bgf_run / bgf_sync
    // launch schedule of the persistent one-level kernels
    BlockXY xy;
    int tile_x = TILE_X, tile_y = TILE_Y, wg_pred = 0, wg_corr = 0;
    // block slots the device arrays hold (>= nblkmem; adapted meshes grow into it)
    int cap = 0;
    // bgf_remesh staging: the new mesh (active, level, 8 neighbours, inv), the
    // remap table and block origins; refine flags
    int* d_mesh2[11] = {nullptr};
    int* d_remap = nullptr;
    double *d_bxo = nullptr, *d_byo = nullptr;
    unsigned char* d_flags = nullptr;
    // block origins (double, cap) for cell positions; rain forcing
    double *d_blkxo = nullptr, *d_blkyo = nullptr;
    double *d_rain_t = nullptr, *d_rain_v = nullptr;
    int rain_n = 0;
    float *d_rframes = nullptr, *d_rnow = nullptr;
    // bed source raster sampled by bgf_remesh for new cells
    float* d_bed = nullptr;
    // boundary segments in the order set, each with its device buffers; the
    // segment of each block slot and the device table (the segments, then the
    // remainder of type aoibnd), rebuilt with the mesh
    std::vector<HostSeg> segs;
    unsigned char* d_bseg = nullptr;
    bgf::BSeg* d_seg = nullptr;
    double zsinit = 0.0;
    std::vector<int> h_nb[8];  // host copy of the neighbours (LeftBot .. BotRight)
    // host copy of the mesh (active list, levels, origins) and the rivers as given
    std::vector<int> h_level;
    std::vector<double> h_xo, h_yo;
    std::vector<double> riv_box, riv_t, riv_q;
    std::vector<int> riv_n;
    // rivers on the device: boxes, series, offsets, areas, block flags
    double *d_rbox = nullptr, *d_rt = nullptr, *d_rq = nullptr, *d_rarea = nullptr;
    int* d_roff = nullptr;
    unsigned char* d_rblk = nullptr;
    int bed_nx = 0, bed_ny = 0;
    double bed_xo = 0, bed_yo = 0, bed_dx = 0;
    // gauge series recorded on the GPU every `gevery` steps (bgf_set_gauges): 16 cells, a ring of
    // GAUGE_CAP samples per gauge and the sample times; nstep counts the steps since they were set
    int* d_gcell = nullptr;
    float* d_gring = nullptr;
    double* d_gtring = nullptr;
    int gevery = 0;
    int nstep = 0;
};

namespace {

void free_handle(bgf_handle h) {
    auto F = [](void* p) { if (p) (void)hipFree(p); };
    F(h->arena);
    if (!h->amr) {
        for (int k = 0; k < 2; k++) { F(h->d_h[k]); F(h->d_u[k]); F(h->d_v[k]); }
        F(h->d_zb); F(h->d_cf); F(h->d_dh); F(h->d_dhu); F(h->d_dhv); F(h->d_ch);
    }
    for (int k = 0; k < 15; k++) F(h->stats.a[k]);
    F(h->d_bed);
    for (HostSeg& g : h->segs) free_seg(g);
    F(h->d_bseg); F(h->d_seg);
    F(h->d_rbox); F(h->d_rt); F(h->d_rq); F(h->d_rarea); F(h->d_roff); F(h->d_rblk);
    F(h->d_rain_t); F(h->d_rain_v); F(h->d_rframes); F(h->d_rnow);
    F(h->d_flags);
    F(h->d_gcell); F(h->d_gring); F(h->d_gtring);
    for (int k = 0; k < 4; k++) if (h->ev[k]) (void)hipEventDestroy(h->ev[k]);
    if (h->graph) (void)hipGraphExecDestroy(h->graph);
    if (h->stream) (void)hipStreamDestroy(h->stream);
    if (h->loop_host) (void)hipHostFree(h->loop_host);
    delete h;
}

// What a handle keeps besides its mesh's buffers: stream, events, pinned memory.
void swap_host_side(bgf_handle a, bgf_handle b) {
    std::swap(a->stream, b->stream);
    std::swap(a->ev, b->ev);
    std::swap(a->loop_host, b->loop_host);
    std::swap(a->back, b->back);
}

bgf_status upload_loop(bgf_handle h, const bgf_loop* loop, double endtime) {
    bgf::LoopState L;
    std::memset(&L, 0, sizeof(L));
    L.nextoutputtime = loop->nextoutputtime;
    L.dt = loop->dt;
    L.dtmax = loop->dtmax;
    L.totaltime = loop->totaltime;
    L.endtime = endtime;
    bgf::set_rain(L, (double)(float)h->p.rain);  // Rain.nowvalue is a float (src/Forcing.h)
    L.rain_t = h->d_rain_t;
    L.rain_v = h->d_rain_v;
    L.rain_n = h->rain_n;
    L.done = loop->totaltime >= endtime ? 1 : 0;
    L.dtmin = h->p.dtmin;
    L.nstep = h->nstep;
    L.gevery = h->gevery;
    L.stats_n = h->stats_n;
    bgf::launch_set_loop(L, h->d_loop, h->stream);
    HIPCHK(hipGetLastError());
    h->loop_at = 0;
    return BGF_OK;
}

// Brings the state back to buffer 0 where it ended in buffer 1 (one-level
// meshes after an odd number of steps); out: see launch_settle.
void enqueue_settle(bgf_handle h, bgf::LoopState* out) {
    const void* src[3] = {h->d_h[1], h->d_u[1], h->d_v[1]};
    void* dst[3] = {h->d_h[0], h->d_u[0], h->d_v[0]};
    bgf::launch_settle(h->prec, h->kp, src, dst, h->d_loop + h->loop_at, out, h->stream);
}

// Waits for the enqueued work, whose last launch wrote the loop state out.
bgf_status finish_loop(bgf_handle h, bgf::LoopState* L) {
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(h->stream));
    *L = *h->loop_host;
    h->stats_n = L->stats_n;
    h->nstep = L->nstep;
    return BGF_OK;
}

// The loop state after `steps` enqueued steps, the state of the domain back in
// buffer 0.
bgf_status download_loop(bgf_handle h, int steps, bgf::LoopState* L) {
    const bool one = !h->amr, odd = one && (steps & 1);
    if (odd) enqueue_settle(h, h->loop_host);
    else bgf::launch_loop_out(h->d_loop + h->loop_at, h->loop_host, h->stream);
    bgf_status s = finish_loop(h, L);
    if (s == BGF_OK && one && !odd && (L->steps_done & 1)) {  // stopped early, after an odd step
        enqueue_settle(h, nullptr);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(h->stream));
    }
    return s;
}

constexpr int GAUGE_CAP = 2048;  // gauge samples kept per gauge

// Output statistics and gauge samples of the state after a step of parity k,
// which leaves its loop state in 1 - k: one-level steps end in buffer 1 - k,
// multi-level steps in buffer 0.
void enqueue_stats(bgf_handle h, int k, int advanced) {
    const int b = h->amr ? 0 : 1 - k;
    const bgf::DevLoop* L = h->d_loop + (1 - k);
    if (h->gevery > 0)
        bgf::launch_gauge_step(h->prec == 0 ? 0 : 1, h->d_h[b], h->d_gcell, L, 1, GAUGE_CAP, h->d_gring, h->d_gtring,
                               h->stream);
    if (!h->stats.mask) return;
    bgf::launch_stats(h->prec == 0 ? 0 : 1, h->kp, h->stats, h->d_h[b], h->d_u[b], h->d_v[b], h->d_zb, L, advanced,
                      h->stream);
}

void fill_buffers(bgf_handle h, int in, void* out_storage) {
    int out = 1 - in;
    if (h->prec == 0) {
        auto* B = (bgf::StepBuffers<double>*)out_storage;
        B->h = (const double*)h->d_h[in]; B->u = (const double*)h->d_u[in]; B->v = (const double*)h->d_v[in];
        B->ho = (double*)h->d_h[out]; B->uo = (double*)h->d_u[out]; B->vo = (double*)h->d_v[out];
        B->zb = (const double*)h->d_zb; B->cf = (const double*)h->d_cf;
        B->dh = (double*)h->d_dh; B->dhu = (double*)h->d_dhu; B->dhv = (double*)h->d_dhv;
        B->ch = nullptr;
    } else {
        auto* B = (bgf::StepBuffers<float>*)out_storage;
        B->h = (const float*)h->d_h[in]; B->u = (const float*)h->d_u[in]; B->v = (const float*)h->d_v[in];
        B->ho = (float*)h->d_h[out]; B->uo = (float*)h->d_u[out]; B->vo = (float*)h->d_v[out];
        B->zb = (const float*)h->d_zb; B->cf = (const float*)h->d_cf;
        B->dh = (float*)h->d_dh; B->dhu = (float*)h->d_dhu; B->dhv = (float*)h->d_dhv;
        B->ch = (float*)h->d_ch;
    }
}

template <class T> void fill_amr_t(bgf_handle h, bgf::AmrBuffers<T>* B) {
    B->h = (T*)h->d_h[0]; B->u = (T*)h->d_u[0]; B->v = (T*)h->d_v[0];
    B->ho = (T*)h->d_h[1]; B->uo = (T*)h->d_u[1]; B->vo = (T*)h->d_v[1];
    B->zb = (T*)h->d_zb; B->cf = (const T*)h->d_cf;
    T** f[8] = {&B->Fhu, &B->Fqux, &B->Su, &B->Fqvx, &B->Fhv, &B->Fqvy, &B->Sv, &B->Fquy};
    for (int k = 0; k < 8; k++) *f[k] = (T*)h->d_amr[2 + k];
    B->hsnap = (T*)h->d_amr[10];
    B->dh = (T*)h->d_dh; B->dhu = (T*)h->d_dhu; B->dhv = (T*)h->d_dhv;
}

void fill_amr_buffers(bgf_handle h, void* storage) {
    if (h->prec == 0) fill_amr_t<double>(h, (bgf::AmrBuffers<double>*)storage);
    else fill_amr_t<float>(h, (bgf::AmrBuffers<float>*)storage);
}

// One step of parity k: from loop state k to 1 - k, and on one-level meshes
// from buffer k to 1 - k.
void enqueue_step(bgf_handle h, int k, int advance_time, hipEvent_t* ev) {
    alignas(16) unsigned char storage[sizeof(bgf::AmrBuffers<double>)];
    bgf::DevLoop *L = h->d_loop + k, *Lnext = h->d_loop + (1 - k);
    if (h->amr) {
        fill_amr_buffers(h, storage);
        bgf::launch_amr_step(h->prec, h->kp, storage, L, Lnext, advance_time, h->stream, ev);
    } else {
        fill_buffers(h, k, storage);
        bgf::launch_step(h->prec, h->kp, storage, L, Lnext, advance_time, h->stream, ev);
    }
    enqueue_stats(h, k, advance_time);
}

// Steps of a captured graph (even: the last leaves the state where the first
// found it).  Shorter runs than two of them launch their kernels directly:
// replaying a graph of two steps was slower than that (1.55 against 1.43 ms
// for 100 steps of 256 x 256 cells), one of eight is faster (1.36 ms), since a
// replay starts about 3 us after the last, and what its capture costs comes
// back only in longer runs.
constexpr int PERIOD = 8;

// Runs of many steps replay a captured HIP graph of PERIOD steps instead of
// relaunching every kernel (the step is launch-bound on small domains and
// multi-level meshes).  The graph holds kernel launches only.
bgf_status graph_steps(bgf_handle h, int nperiods) {
    if (!h->graph) {
        hipGraph_t g = nullptr;
        HIPCHK(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
        for (int k = 0; k < PERIOD; k++) enqueue_step(h, k & 1, 1, nullptr);
        HIPCHK(hipStreamEndCapture(h->stream, &g));
        hipError_t e = hipGraphInstantiate(&h->graph, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
            h->graph = nullptr;
            return fail(BGF_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
        }
    }
    for (int k = 0; k < nperiods; k++) HIPCHK(hipGraphLaunch(h->graph, h->stream));
    return BGF_OK;
}

bgf_status enqueue_steps(bgf_handle h, int nsteps, int advance_time) {
    h->loop_at = nsteps & 1;
    if (advance_time == 1 && !h->timing && h->use_graph && nsteps >= 2 * PERIOD) {
        bgf_status s = graph_steps(h, nsteps / PERIOD);
        if (s != BGF_OK) return s;
        nsteps %= PERIOD;
    }
    for (int k = 0; k < nsteps; k++) {
        enqueue_step(h, k & 1, advance_time, h->timing ? h->ev : nullptr);
        if (h->timing) {
            HIPCHK(hipEventSynchronize(h->ev[3]));
            float a = 0, b = 0, c = 0;
            HIPCHK(hipEventElapsedTime(&a, h->ev[0], h->ev[1]));
            HIPCHK(hipEventElapsedTime(&b, h->ev[1], h->ev[2]));
            HIPCHK(hipEventElapsedTime(&c, h->ev[2], h->ev[3]));
            h->t_pred += a; h->t_red += b; h->t_corr += c; h->t_n += 1;
        }
    }
    HIPCHK(hipGetLastError());
    return BGF_OK;
}

}  // namespace

extern "C" {

const char* bgf_last_error(void) { return g_err.c_str(); }

const char* bgf_version(void) { return "bgflood_amd 0.1 (gfx950)"; }

int bgf_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

}  // extern "C"

namespace {

// Mesh validation.  One-level meshes (every side a boundary or one same-level
// neighbour) run the fused kernels; others the multi-level ones, which need
// neighbour levels within one of each other (2:1 balance).
struct MeshInfo {
    bool multilevel = false;
    int minlev = 1 << 30, maxlev = -(1 << 30);
    std::vector<int> inv;
};

bgf_status check_mesh(const bgf_param* p, const bgf_blocks* b, MeshInfo& m) {
    const int nblk = p->nblk, nbm = p->nblkmem;
    m.inv.assign(nbm, -1);
    for (int ibl = 0; ibl < nblk; ibl++) {
        int ib = b->active[ibl];
        if (ib < 0 || ib >= nbm) return fail(BGF_ERR_INVALID_ARG, "active block index out of range");
        if (m.inv[ib] >= 0) return fail(BGF_ERR_INVALID_ARG, "block listed twice in active");
        m.inv[ib] = ibl;
        m.minlev = std::min(m.minlev, b->level[ib]);
        m.maxlev = std::max(m.maxlev, b->level[ib]);
    }
    for (int ibl = 0; ibl < nblk; ibl++) {
        int ib = b->active[ibl];
        const int* pairs[4][2] = {{b->LeftBot, b->LeftTop}, {b->RightBot, b->RightTop},
                                  {b->TopLeft, b->TopRight}, {b->BotLeft, b->BotRight}};
        for (auto& pr : pairs) {
            int n0 = pr[0][ib], n1 = pr[1][ib];
            if (n0 < 0 || n0 >= nbm || n1 < 0 || n1 >= nbm) return fail(BGF_ERR_INVALID_ARG, "neighbour out of range");
            if (m.inv[n0] < 0 || m.inv[n1] < 0) return fail(BGF_ERR_INVALID_ARG, "neighbour is not an active block");
            for (int n : {n0, n1})
                if (std::abs(b->level[n] - b->level[ib]) > 1)
                    return fail(BGF_ERR_INVALID_ARG, "neighbour levels differ by more than one");
            if (n0 != n1 || (n0 != ib && b->level[n0] != b->level[ib])) m.multilevel = true;
        }
    }
    if (m.minlev != m.maxlev) m.multilevel = true;
    // spherical grids run on the general (multi-level) kernels, which take per-row metric terms
    if (p->spherical) m.multilevel = true;
    return BGF_OK;
}

// Per-block metric terms of a spherical mesh, uploaded to the handle.
bool upload_metric(bgf_handle h, const bgf_param* p, const bgf_blocks* b, int nbm) {
    if (h->prec == 0) {
        std::vector<double> M = metric_table<double>(p, b, nbm);
        return hipMemcpy(h->d_metric, M.data(), sizeof(double) * M.size(), hipMemcpyHostToDevice) == hipSuccess;
    }
    std::vector<float> M = metric_table<float>(p, b, nbm);
    return hipMemcpy(h->d_metric, M.data(), sizeof(float) * M.size(), hipMemcpyHostToDevice) == hipSuccess;
}

// The blocks of the handle's current mesh that the multi-level step advances
// after the others (fix_blocks), for the current boundary segments.
bgf_status setup_fix(bgf_handle h) {
    if (!h->amr) return BGF_OK;
    bool all = false, odd = false;
    const std::vector<int> list =
        fix_blocks(h->active.data(), h->nblk, h->h_level.data(), h->h_nb, h->kp.bopen != 0, all, odd);
    if (!list.empty()) HIPCHK(hipMemcpy(h->d_fix, list.data(), sizeof(int) * list.size(), hipMemcpyHostToDevice));
    h->kp.fix = h->d_fix;
    h->kp.nfix = (int)list.size();
    h->kp.fix_all = all ? 1 : 0;
    h->kp.odd = odd ? 1 : 0;
    return BGF_OK;
}

// The boundary segments on the handle's current mesh: the segment of each
// boundary block (assign_segments; the side strips from the mesh's extent,
// XParam.xmax = Param.xo + the right edge of the easternmost block as
// src/ReadInput.cu:1282-1283 sets it, and epsbnd = calcres(dx, initlevel) with
// initlevel 0), and the device table with the remainder (type aoibnd) last.
// Without segments every boundary face is of type aoibnd and nothing is kept.
bgf_status segment_table(bgf_handle h) {
    bgf::KParams& kp = h->kp;
    if (h->d_bseg) (void)hipFree(h->d_bseg);
    if (h->d_seg) (void)hipFree(h->d_seg);
    h->d_bseg = nullptr;
    h->d_seg = nullptr;
    kp.bseg = nullptr;
    kp.seg = nullptr;
    kp.nseg = kp.bmapmax = kp.bopen = 0;
    if (h->graph) {
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    if (h->segs.empty()) return BGF_OK;
    const bgf_param& p = h->p;
    auto inT = [&](double v) { return h->prec == 0 ? v : (double)(float)v; };  // XBlock.xo is a T
    double xmax = -1e300, ymax = -1e300;
    for (int ib : h->active) {
        const double levdx = level_dx(p.dx, h->h_level[ib]);
        xmax = std::max(xmax, p.xo + inT(h->h_xo[ib]) + (BW - 0.5) * levdx);
        ymax = std::max(ymax, p.yo + inT(h->h_yo[ib]) + (BW - 0.5) * levdx);
    }
    std::vector<Polygon> polys;
    for (const HostSeg& g : h->segs)
        polys.push_back(g.side >= 0 ? side_strip(g.side, p.xo, xmax, p.yo, ymax, p.dx) : g.poly);
    const std::vector<unsigned char> bseg =
        h->prec == 0 ? assign_segments<double>(p, h->active, h->h_level, h->h_xo, h->h_yo, h->h_nb, polys, h->cap)
                     : assign_segments<float>(p, h->active, h->h_level, h->h_xo, h->h_yo, h->h_nb, polys, h->cap);
    std::vector<bgf::BSeg> tab;
    int open = 0, mapmax = 0;
    for (const HostSeg& g : h->segs) {
        bgf::BSeg b{};
        b.type = g.type == 4 ? 1 : g.type;  // type 4 acts as type 1 in engine 2's flux boundary
        b.n = (int)g.t.size();
        b.t = g.d_series;
        b.z = g.d_series ? g.d_series + b.n : nullptr;
        b.zs0 = h->zsinit;
        b.nx = g.nx; b.ny = g.ny; b.nt = g.nt;
        b.xo = g.xo; b.yo = g.yo; b.dx = g.dx; b.dy = g.dy; b.to = g.to; b.tdt = g.tdt;
        if (g.ext_now) {
            b.now = const_cast<float*>(g.ext_now);
        } else if (g.nt == 1) {
            b.now = g.d_frames;
        } else if (g.nt >= 2) {
            b.frames = g.d_frames;
            b.now = g.d_now;
            mapmax = std::max(mapmax, g.nx * g.ny);
        }
        b.on = b.n >= 2 || b.now ? 1 : 0;
        open |= b.type >= 2 ? 1 : 0;
        tab.push_back(b);
    }
    bgf::BSeg rem{};
    rem.type = p.aoibnd;
    rem.zs0 = h->zsinit;
    tab.push_back(rem);
    HIPCHK(hipMalloc((void**)&h->d_bseg, bseg.size()));
    HIPCHK(hipMalloc((void**)&h->d_seg, sizeof(bgf::BSeg) * tab.size()));
    HIPCHK(hipMemcpy(h->d_bseg, bseg.data(), bseg.size(), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(h->d_seg, tab.data(), sizeof(bgf::BSeg) * tab.size(), hipMemcpyHostToDevice));
    kp.bseg = h->d_bseg;
    kp.seg = h->d_seg;
    kp.nseg = (int)tab.size();
    kp.bopen = open;
    kp.bmapmax = mapmax;
    return BGF_OK;
}

// The segments and the blocks whose advance waits for them, which the stage
// takes from kp.bopen: the two agree also where the table could not be made.
bgf_status setup_segments(bgf_handle h) {
    const bgf_status s = segment_table(h), f = setup_fix(h);
    return s != BGF_OK ? s : f;
}

// The rivers on the handle's current mesh (InitialConditions.cu:346-445):
// each river's discharge cells are those whose box, formed in double,
// overlaps the river's; its discharge area sums their areas; rivers without
// a cell are dropped, as the reference drops them; the blocks holding a
// discharge cell of any river are flagged.  Uploads everything the kernels read.
bgf_status setup_rivers(bgf_handle h) {
    auto F = [](auto*& p) { if (p) (void)hipFree(p); p = nullptr; };
    F(h->d_rbox); F(h->d_rt); F(h->d_rq); F(h->d_rarea); F(h->d_roff); F(h->d_rblk);
    bgf::KParams& kp = h->kp;
    kp.nriver = 0;
    kp.rbox = kp.rt = kp.rq = kp.rarea = nullptr;
    kp.roff = nullptr;
    kp.rblk = nullptr;
    const int nr = (int)h->riv_n.size();
    if (nr == 0) return BGF_OK;
    const bgf_param& p = h->p;
    std::vector<double> box, tt, qq, area;
    std::vector<int> off(1, 0);
    std::vector<unsigned char> blk(h->cap, 0);
    int o = 0;
    for (int r = 0; r < nr; r++) {
        const double* bx = &h->riv_box[4 * r];
        double a = 0.0;
        std::vector<int> hit;
        for (int ib : h->active) {
            const double levdx = level_dx(p.dx, h->h_level[ib]), levdelta = level_dx(p.delta, h->h_level[ib]);
            bool any = false;
            for (int j = 0; j < BW; j++)
                for (int i = 0; i < BW; i++) {
                    const double xi = p.xo + h->h_xo[ib] + i * levdx, yi = p.yo + h->h_yo[ib] + j * levdx;
                    const double xl = xi - 0.5 * levdx, yb = yi - 0.5 * levdx, xr = xi + 0.5 * levdx,
                                 yt = yi + 0.5 * levdx;
                    if (bx[0] <= xr && bx[1] >= xl && bx[2] <= yt && bx[3] >= yb) {
                        a = a + (p.spherical ? cell_area_sphere(p.Radius, xi, yi, levdx) : levdelta * levdelta);
                        any = true;
                    }
                }
            if (any) hit.push_back(ib);
        }
        const int n = h->riv_n[r];
        if (a == 0.0) {
            o += n;
            continue;  // outside the active domain
        }
        for (int ib : hit) blk[ib] = 1;
        box.insert(box.end(), bx, bx + 4);
        tt.insert(tt.end(), h->riv_t.begin() + o, h->riv_t.begin() + o + n);
        qq.insert(qq.end(), h->riv_q.begin() + o, h->riv_q.begin() + o + n);
        off.push_back(off.back() + n);
        area.push_back(a);
        o += n;
    }
    const int nk = (int)area.size();
    if (nk == 0) return BGF_OK;
    bool ok = hipMalloc((void**)&h->d_rbox, sizeof(double) * box.size()) == hipSuccess &&
              hipMalloc((void**)&h->d_rt, sizeof(double) * tt.size()) == hipSuccess &&
              hipMalloc((void**)&h->d_rq, sizeof(double) * qq.size()) == hipSuccess &&
              hipMalloc((void**)&h->d_rarea, sizeof(double) * nk) == hipSuccess &&
              hipMalloc((void**)&h->d_roff, sizeof(int) * (nk + 1)) == hipSuccess &&
              hipMalloc((void**)&h->d_rblk, h->cap) == hipSuccess;
    ok = ok && hipMemcpy(h->d_rbox, box.data(), sizeof(double) * box.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(h->d_rt, tt.data(), sizeof(double) * tt.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(h->d_rq, qq.data(), sizeof(double) * qq.size(), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(h->d_rarea, area.data(), sizeof(double) * nk, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(h->d_roff, off.data(), sizeof(int) * (nk + 1), hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(h->d_rblk, blk.data(), h->cap, hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) return fail(BGF_ERR_HIP, "river upload failed");
    kp.nriver = nk;
    kp.rbox = h->d_rbox; kp.rt = h->d_rt; kp.rq = h->d_rq; kp.rarea = h->d_rarea;
    kp.roff = h->d_roff; kp.rblk = h->d_rblk;
    return BGF_OK;
}

// The device arrays of a new handle for h->cap block slots, cleared.  What is
// small goes into one allocation, and on multi-level meshes everything: such a
// handle grows with its mesh (bgf_remesh re-creates it), and an allocation of a
// cells' array takes 0.28 ms and its release 0.26 ms (5 MB each) wherever the
// runtime has no freed piece of its size at hand, so that a growth of 22 of
// them took from 3.8 to 6.8 ms as it came.
bool device_room(bgf_handle h) {
    const size_t cap = h->cap, cells = h->es * cap * BS;
    const bool all = h->amr;
    std::vector<std::pair<void**, size_t>> parts, own;
    auto put = [&](auto*& ptr, size_t bytes) { parts.push_back({(void**)&ptr, bytes}); };
    auto put_cells = [&](void*& ptr) { (all ? parts : own).push_back({&ptr, cells}); };
    put(h->d_active, sizeof(int) * cap);
    put(h->d_level, sizeof(int) * cap);
    for (int k = 0; k < 8; k++) put(h->d_nb[k], sizeof(int) * cap);
    put(h->d_volpart, sizeof(double) * cap);
    put(h->d_volout, sizeof(double));
    put(h->d_loop, 2 * sizeof(bgf::DevLoop));
    put(h->d_blkxo, sizeof(double) * cap);
    put(h->d_blkyo, sizeof(double) * cap);
    for (int k = 0; k < 2; k++) {
        put_cells(h->d_h[k]);
        put_cells(h->d_u[k]);
        put_cells(h->d_v[k]);
    }
    for (void** a : {&h->d_zb, &h->d_cf, &h->d_dh, &h->d_dhu, &h->d_dhv}) put_cells(*a);
    if (h->p.spherical) put(h->d_metric, h->es * cap * bgf::METRIC_STRIDE);
    if (all) {
        put(h->d_inv, sizeof(int) * cap);
        put(h->d_nbr, sizeof(int) * bgf::NBR * cap);
        put(h->d_rcell, sizeof(int4) * bgf::RECIPES * cap);
        put(h->d_rmeta, sizeof(int2) * bgf::RECIPES * cap);
        put(h->d_fix, sizeof(int) * cap);
        for (int k = 0; k < 11; k++) put_cells(h->d_amr[k]);
        for (int k = 0; k < 11; k++) put(h->d_mesh2[k], sizeof(int) * cap);
        put(h->d_remap, sizeof(int) * 5 * cap);
        put(h->d_bxo, sizeof(double) * cap);
        put(h->d_byo, sizeof(double) * cap);
    } else {  // the persistent kernels' order, records and queues
        put(h->d_order, sizeof(int) * cap);
        put(h->d_rec, sizeof(int) * 8 * cap);
        put(h->d_queue, sizeof(int) * 2 * bgf::NXCD * bgf::QSTRIDE);
        if (h->prec == BGF_FP32_COMP) put_cells(h->d_ch);
    }
    auto up = [](size_t n) { return (n + 4095) / 4096 * 4096; };  // as allocations of their own are aligned
    size_t bytes = 0;
    for (auto& q : parts) bytes += up(q.second);
    own.push_back({&h->arena, bytes});
    for (auto& q : own)
        if (hipMalloc(q.first, q.second) != hipSuccess || hipMemset(*q.first, 0, q.second) != hipSuccess) return false;
    unsigned char* at = (unsigned char*)h->arena;
    for (auto& q : parts) {
        *q.first = at;
        at += up(q.second);
    }
    return true;
}

// bgf_create with device arrays for cap >= nblkmem block slots.  from: a handle
// that the new one replaces, whose stream, events and pinned memory it takes.
bgf_status create_handle(const bgf_param* p, const bgf_blocks* b, int cap, bgf_handle* out, bgf_handle from = nullptr) {
    if (!out || !b) return fail(BGF_ERR_INVALID_ARG, "null argument");
    *out = nullptr;
    bgf_status s = check_param(p);
    if (s != BGF_OK) return s;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(BGF_ERR_NO_DEVICE, "no HIP device");
    const int nblk = p->nblk, nbm = p->nblkmem;
    if (cap < nbm) cap = nbm;
    if (!block_bytes_ok(cap, p->precision))
        return fail(BGF_ERR_UNSUPPORTED, "block capacity " + std::to_string(cap) + " above the 32-bit offset limit");
    MeshInfo mi;
    s = check_mesh(p, b, mi);
    if (s != BGF_OK) return s;
    const bool multilevel = mi.multilevel;
    const int minlev = mi.minlev, maxlev = mi.maxlev;
    std::vector<int>& inv = mi.inv;
    auto* h = new bgf_handle_s();
    if (from) swap_host_side(h, from);
    auto drop = [&](bgf_status e) {
        if (from) swap_host_side(h, from);
        free_handle(h);
        return e;
    };
    h->p = *p;
    h->prec = p->precision;
    h->es = p->precision == 0 ? sizeof(double) : sizeof(float);
    h->nblk = nblk;
    h->nblkmem = nbm;
    h->cap = cap;
    h->S = (size_t)nbm * BS;
    const size_t SA = (size_t)cap * BS;  // values per allocated array
    h->active.assign(b->active, b->active + nblk);
    h->h_level.assign(b->level, b->level + nbm);
    h->h_xo.assign(b->xo, b->xo + nbm);
    h->h_yo.assign(b->yo, b->yo + nbm);
    {
        const int* nb[8] = {b->LeftBot, b->LeftTop, b->RightBot, b->RightTop, b->TopLeft, b->TopRight, b->BotLeft, b->BotRight};
        for (int k = 0; k < 8; k++) h->h_nb[k].assign(nb[k], nb[k] + nbm);
    }
    h->amr = multilevel;
    bool ok = device_room(h);
    if (!h->loop_host)
        ok = ok && hipHostMalloc((void**)&h->loop_host, sizeof(bgf::LoopState), hipHostMallocDefault) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        return drop(fail(BGF_ERR_OOM, "device allocation failed"));
    }
    const int* nbs[8] = {b->LeftBot, b->LeftTop, b->RightBot, b->RightTop, b->TopLeft, b->TopRight, b->BotLeft, b->BotRight};
    h->xy = block_xy(b, nblk, p->dx);
    bool cp = hipMemcpy(h->d_active, b->active, sizeof(int) * nblk, hipMemcpyHostToDevice) == hipSuccess;
    if (!multilevel) {
        std::vector<int> order = processing_order(h->xy);
        cp = cp && hipMemcpy(h->d_order, order.data(), sizeof(int) * nblk, hipMemcpyHostToDevice) == hipSuccess;
    }
    cp = cp && hipMemcpy(h->d_level, b->level, sizeof(int) * nbm, hipMemcpyHostToDevice) == hipSuccess;
    cp = cp && hipMemcpy(h->d_blkxo, b->xo, sizeof(double) * nbm, hipMemcpyHostToDevice) == hipSuccess;
    cp = cp && hipMemcpy(h->d_blkyo, b->yo, sizeof(double) * nbm, hipMemcpyHostToDevice) == hipSuccess;
    for (int k = 0; k < 8; k++) cp = cp && hipMemcpy(h->d_nb[k], nbs[k], sizeof(int) * nbm, hipMemcpyHostToDevice) == hipSuccess;
    if (p->spherical) cp = cp && upload_metric(h, p, b, nbm);
    if (multilevel) {
        cp = cp && hipMemcpy(h->d_inv, inv.data(), sizeof(int) * nbm, hipMemcpyHostToDevice) == hipSuccess;
    }
    if (!from) {
        cp = cp && hipStreamCreate(&h->stream) == hipSuccess;
        for (int k = 0; k < 4; k++) cp = cp && hipEventCreate(&h->ev[k]) == hipSuccess;
    }
    if (!cp) return drop(fail(BGF_ERR_HIP, "device upload failed"));
    bgf::KParams& kp = h->kp;
    kp.g = p->g; kp.eps = p->eps; kp.CFL = p->CFL; kp.theta = p->theta;
    kp.delta0 = p->delta;
    kp.delta = minlev < 0 ? p->delta * (1 << -minlev) : p->delta / (1 << minlev);  // one-level kernels
    kp.fc = p->precision == 0 ? coriolis<double>(p->lat) : coriolis<float>(p->lat);
    kp.mask = p->mask;
    kp.rain_mmh = (double)(float)p->rain;  // Rain.nowvalue is a float (src/Forcing.h)
    kp.frictionmodel = p->frictionmodel;
    kp.aoibnd = p->aoibnd;
    kp.ForceMassConserve = p->ForceMassConserve;
    kp.rain_on = p->rain_on;
    kp.nblk = nblk;
    kp.wetdryfix = p->wetdryfix;
    kp.minlevel = minlev;
    kp.maxlevel = maxlev;
    // BGF_WG_PER_CU="p,c" caps the persistent workgroups per CU of the
    // predictor and the corrector (a tuning override; default: occupancy).
    if (const char* e = std::getenv("BGF_WG_PER_CU")) std::sscanf(e, "%d,%d", &h->wg_pred, &h->wg_corr);
    if (const char* e = std::getenv("BGF_GRAPH")) h->use_graph = std::atoi(e) != 0;
    kp.grid_pred = bgf::persistent_grid(h->prec, 0, nblk, h->wg_pred);
    kp.grid_corr = bgf::persistent_grid(h->prec, 1, nblk, h->wg_corr);
    if (kp.grid_pred <= 0 || kp.grid_corr <= 0) return drop(fail(BGF_ERR_HIP, "occupancy query failed"));
    kp.active = h->d_active;
    kp.order = h->d_order;
    kp.rec = h->d_rec;
    kp.queue = h->d_queue;
    kp.LeftBot = h->d_nb[0];
    kp.RightBot = h->d_nb[2];
    kp.TopLeft = h->d_nb[4];
    kp.BotLeft = h->d_nb[6];
    kp.level = h->d_level;
    kp.LeftTop = h->d_nb[1];
    kp.RightTop = h->d_nb[3];
    kp.TopRight = h->d_nb[5];
    kp.BotRight = h->d_nb[7];
    kp.inv = h->d_inv;
    kp.metric = h->d_metric;
    kp.spherical = p->spherical;
    kp.xo = p->xo;
    kp.yo = p->yo;
    kp.dx = p->dx;
    kp.bxo = h->d_blkxo;
    kp.byo = h->d_blkyo;
    kp.nbr = h->d_nbr;
    kp.rcell = h->d_rcell;
    kp.rmeta = h->d_rmeta;
    if (multilevel) bgf::launch_amr_nbr(kp, h->d_nbr, nbm, h->d_rcell, h->d_rmeta, h->stream);
    else bgf::launch_records(kp, h->d_rec, h->stream);
    if (hipGetLastError() != hipSuccess) return drop(fail(BGF_ERR_HIP, "block records launch failed"));
    s = setup_fix(h);
    if (s != BGF_OK) return drop(s);
    *out = h;
    g_err.clear();
    return BGF_OK;
}

// A roughness that is one value over the active cells (a constant Param.cf, the usual case) is
// passed to the one-level corrector as that value instead of being read per cell; not once the
// caller holds the device array (bgf_device_array), which it may change.  cf: host array.
void detect_uniform_cf(bgf_handle h, const void* cf) {
    int uni = !h->cf_shared;
    double val = 0.0;
    for (int ibl = 0; uni && ibl < h->nblk; ibl++) {
        const int ib = h->active[ibl];
        for (int j = 0; uni && j < BW; j++)
            for (int i = 0; i < BW; i++) {
                const size_t n = (size_t)memloc(i, j, ib);
                const double c = h->prec == 0 ? ((const double*)cf)[n] : (double)((const float*)cf)[n];
                if (ibl == 0 && i == 0 && j == 0) val = c;
                else if (!(c == val) || std::signbit(c) != std::signbit(val)) { uni = 0; break; }
            }
    }
    if (uni != h->kp.cf_uniform || (uni && val != h->kp.cf_value)) {
        h->kp.cf_uniform = uni;
        h->kp.cf_value = uni ? val : 0.0;
        if (h->graph) {  // the captured launches carry the old parameters
            (void)hipGraphExecDestroy(h->graph);
            h->graph = nullptr;
        }
    }
}

}  // namespace

extern "C" {

bgf_status bgf_create(const bgf_param* p, const bgf_blocks* b, bgf_handle* out) {
    return create_handle(p, b, p ? p->nblkmem : 0, out);
}

bgf_status bgf_destroy(bgf_handle h) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    (void)hipStreamSynchronize(h->stream);
    free_handle(h);
    return BGF_OK;
}

bgf_status bgf_set_state(bgf_handle h, const void* zb, const void* hh, const void* u, const void* v, const void* cf) {
    if (!h || !zb || !hh || !u || !v || !cf) return fail(BGF_ERR_INVALID_ARG, "null argument");
    size_t bytes = h->es * h->S;
    HIPCHK(hipMemcpyAsync(h->d_zb, zb, bytes, hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->d_h[0], hh, bytes, hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->d_u[0], u, bytes, hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->d_v[0], v, bytes, hipMemcpyHostToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->d_cf, cf, bytes, hipMemcpyHostToDevice, h->stream));
    if (h->d_ch) HIPCHK(hipMemsetAsync(h->d_ch, 0, h->es * h->S, h->stream));
    detect_uniform_cf(h, cf);
    if (h->amr) {
        // halo of the bed, as InitzbHalo (src/InitialConditions.cu:135-147)
        bgf::launch_amr_fill(h->prec == 0 ? 0 : 1, h->kp, h->d_zb, h->stream);
        HIPCHK(hipGetLastError());
    }
    HIPCHK(hipStreamSynchronize(h->stream));
    h->state_set = true;
    return BGF_OK;
}

bgf_status bgf_get_state(bgf_handle h, void* zs, void* hh, void* u, void* v) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    void* const dst[4] = {zs, hh, u, v};
    return read_back(*h->back, h->prec, h->active, h->nblk, 0, h->d_active, h->d_zb, h->d_h[0], h->d_u[0], h->d_v[0], dst,
                     h->stream);
}

bgf_status bgf_init_dt(bgf_handle h, double dtinit, bgf_loop* loop) {
    if (!h || !loop) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (!h->state_set) return fail(BGF_ERR_STATE, "state not set");
    bgf_loop L = *loop;
    // src/Mainloop.cu:524-536
    if (dtinit > 0) L.dtmax = dtinit / 1.5;
    else L.dtmax = (h->p.maxlevel < 0 ? h->p.delta * (1 << -h->p.maxlevel) : h->p.delta / (1 << h->p.maxlevel)) /
                   std::sqrt(h->p.g * 10.0);
    bgf_status s = upload_loop(h, &L, 1e300);
    if (s != BGF_OK) return s;
    bgf::launch_init_dt(h->prec, h->kp, h->d_h[0], h->d_loop, h->stream);
    HIPCHK(hipGetLastError());
    bgf::LoopState D;
    s = download_loop(h, 0, &D);
    if (s != BGF_OK) return s;
    loop->dtmax = D.dt;
    return BGF_OK;
}

bgf_status bgf_step(bgf_handle h, bgf_loop* loop) {
    if (!h || !loop) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (!h->state_set) return fail(BGF_ERR_STATE, "state not set");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    bgf_status s = upload_loop(h, loop, 1e300);
    if (s != BGF_OK) return s;
    s = enqueue_steps(h, 1, 0);
    if (s != BGF_OK) return s;
    bgf::LoopState D;
    s = download_loop(h, 1, &D);  // cleanup: evolv_o -> evolv (src/FlowGPU.cu:282)
    if (s != BGF_OK) return s;
    loop->dt = D.dt;
    loop->dtmax = D.dtmax;
    if (D.bad) return fail(BGF_ERR_NONFINITE_DT, "non-finite or non-positive time step");
    return BGF_OK;
}

bgf_status bgf_run_async(bgf_handle h, const bgf_loop* loop, int nsteps, double endtime) {
    if (!h || !loop || nsteps < 0) return fail(BGF_ERR_INVALID_ARG, "bad argument");
    if (!h->state_set) return fail(BGF_ERR_STATE, "state not set");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    bgf_status s = upload_loop(h, loop, endtime);
    if (s != BGF_OK) return s;
    s = enqueue_steps(h, nsteps, 1);
    if (s != BGF_OK) return s;
    h->pending_steps = nsteps > 0 ? nsteps : -1;
    return BGF_OK;
}

bgf_status bgf_sync(bgf_handle h, bgf_loop* loop) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (!h->pending_steps) return fail(BGF_ERR_STATE, "nothing pending");
    bgf::LoopState D;
    const int steps = h->pending_steps > 0 ? h->pending_steps : 0;
    h->pending_steps = 0;
    bgf_status s = download_loop(h, steps, &D);
    if (s != BGF_OK) return s;
    h->last_steps = D.steps_done;
    if (loop) {
        loop->dt = D.dt;
        loop->dtmax = D.dtmax;
        loop->totaltime = D.totaltime;
    }
    if (D.bad) return fail(BGF_ERR_NONFINITE_DT, "non-finite or non-positive time step");
    if (D.crashed)
        return fail(BGF_ERR_CRASHED, "Model CRASHED: time step " + std::to_string(D.dt) + " below dtmin " +
                                         std::to_string(h->p.dtmin) + " at t = " + std::to_string(D.totaltime));
    return BGF_OK;
}

bgf_status bgf_run(bgf_handle h, bgf_loop* loop, int nsteps, double endtime) {
    bgf_status s = bgf_run_async(h, loop, nsteps, endtime);
    if (s != BGF_OK) return s;
    return bgf_sync(h, loop);
}

bgf_status bgf_set_state_device(bgf_handle h, const void* zb, const void* hh, const void* u, const void* v,
                                const void* cf) {
    if (!h || !zb || !hh || !u || !v || !cf) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    for (const void* q : {zb, hh, u, v, cf})
        if (!device_accessible(q)) return fail(BGF_ERR_INVALID_ARG, "bgf_set_state_device: arrays must be device memory");
    const size_t bytes = h->es * h->S;
    HIPCHK(hipMemcpyAsync(h->d_zb, zb, bytes, hipMemcpyDeviceToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->d_h[0], hh, bytes, hipMemcpyDeviceToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->d_u[0], u, bytes, hipMemcpyDeviceToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->d_v[0], v, bytes, hipMemcpyDeviceToDevice, h->stream));
    HIPCHK(hipMemcpyAsync(h->d_cf, cf, bytes, hipMemcpyDeviceToDevice, h->stream));
    if (h->d_ch) HIPCHK(hipMemsetAsync(h->d_ch, 0, h->es * h->S, h->stream));
    std::vector<unsigned char> cfh(bytes);
    HIPCHK(hipMemcpyAsync(cfh.data(), cf, bytes, hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    detect_uniform_cf(h, cfh.data());
    if (h->amr) {
        bgf::launch_amr_fill(h->prec == 0 ? 0 : 1, h->kp, h->d_zb, h->stream);
        HIPCHK(hipGetLastError());
    }
    HIPCHK(hipStreamSynchronize(h->stream));
    h->state_set = true;
    return BGF_OK;
}

bgf_status bgf_step_device(bgf_handle h, void* hh, void* zs, void* u, void* v, const void* zb, bgf_loop* loop) {
    if (!h || !hh || !zs || !u || !v || !loop) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (!h->state_set) return fail(BGF_ERR_STATE, "state not set");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    for (const void* q : {(const void*)hh, (const void*)zs, (const void*)u, (const void*)v})
        if (!device_accessible(q)) return fail(BGF_ERR_INVALID_ARG, "bgf_step_device: arrays must be device memory");
    if (zb && !device_accessible(zb)) return fail(BGF_ERR_INVALID_ARG, "bgf_step_device: zb must be device memory");
    const int pr = h->prec == 0 ? 0 : 1;
    if (zb) {
        HIPCHK(hipMemcpyAsync(h->d_zb, zb, h->es * h->S, hipMemcpyDeviceToDevice, h->stream));
        if (h->amr) bgf::launch_amr_fill(pr, h->kp, h->d_zb, h->stream);
    }
    bgf_status s = upload_loop(h, loop, 1e300);
    if (s != BGF_OK) return s;
    const void* caller[3] = {hh, u, v};
    if (h->amr) {
        // the multi-level step works in place on its own arrays (halos included): bring the
        // caller's state in, step, and hand it back
        void* mine[3] = {h->d_h[0], h->d_u[0], h->d_v[0]};
        bgf::launch_import(pr, h->kp, caller, mine, h->stream);
        s = enqueue_steps(h, 1, 0);
        if (s != BGF_OK) return s;
        const void* res[3] = {h->d_h[0], h->d_u[0], h->d_v[0]};
        void* out[4] = {hh, zs, u, v};
        bgf::launch_export(pr, h->kp, res, h->d_zb, out, nullptr, h->d_loop + h->loop_at, h->loop_host, h->stream);
    } else {
        // the one-level kernels read the step-start state straight from the caller's arrays and
        // write U^{n+1} into the handle's second buffer, which then goes back to the caller (the
        // reference's cleanup copy evolv_o -> evolv, src/FlowGPU.cu:282) and into the handle's
        // first buffer (its own state for volume, statistics and later runs)
        alignas(16) unsigned char storage[sizeof(bgf::AmrBuffers<double>)];
        fill_buffers(h, 0, storage);
        if (h->prec == 0) {
            auto* B = (bgf::StepBuffers<double>*)storage;
            B->h = (const double*)hh; B->u = (const double*)u; B->v = (const double*)v;
        } else {
            auto* B = (bgf::StepBuffers<float>*)storage;
            B->h = (const float*)hh; B->u = (const float*)u; B->v = (const float*)v;
        }
        bgf::launch_step(h->prec, h->kp, storage, h->d_loop, h->d_loop + 1, 0, h->stream, nullptr);
        enqueue_stats(h, 0, 0);
        h->loop_at = 1;
        const void* res[3] = {h->d_h[1], h->d_u[1], h->d_v[1]};
        void* out[4] = {hh, zs, u, v};
        void* keep[3] = {h->d_h[0], h->d_u[0], h->d_v[0]};
        bgf::launch_export(pr, h->kp, res, h->d_zb, out, keep, h->d_loop + h->loop_at, h->loop_host, h->stream);
    }
    bgf::LoopState D;
    s = finish_loop(h, &D);
    if (s != BGF_OK) return s;
    loop->dt = D.dt;
    loop->dtmax = D.dtmax;
    if (D.bad) return fail(BGF_ERR_NONFINITE_DT, "non-finite or non-positive time step");
    return BGF_OK;
}

bgf_status bgf_set_rain_rate(bgf_handle h, double rain_mmh) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (!std::isfinite(rain_mmh)) return fail(BGF_ERR_INVALID_ARG, "rain rate must be finite");
    h->p.rain = rain_mmh;
    if (!h->p.rain_on) {
        h->p.rain_on = 1;
        h->kp.rain_on = 1;
        if (h->graph) {  // the captured launches carry the old parameters
            (void)hipGraphExecDestroy(h->graph);
            h->graph = nullptr;
        }
    }
    return BGF_OK;
}

bgf_status bgf_set_rain_map_device(bgf_handle h, int nx, int ny, double xo, double yo, double dx,
                                   const float* now_g) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (now_g && (nx < 2 || ny < 2 || !(dx > 0)))
        return fail(BGF_ERR_INVALID_ARG, "a rain map needs nx, ny >= 2 and dx > 0");
    HIPCHK(hipStreamSynchronize(h->stream));
    (void)hipFree(h->d_rframes);
    (void)hipFree(h->d_rnow);
    h->d_rframes = h->d_rnow = nullptr;
    bgf::KParams& kp = h->kp;
    kp.rframes = nullptr;
    kp.rnow = nullptr;
    kp.rnframes = 0;
    if (now_g) {
        // one frame, read in place: no interpolation in time here (the caller's updateforcing did it)
        kp.rframes = now_g;
        kp.rnow = const_cast<float*>(now_g);
        kp.rnx = nx; kp.rny = ny; kp.rnframes = 1;
        kp.rxo = xo; kp.ryo = yo; kp.rdx = dx; kp.rt0 = 0.0; kp.rdtf = 1.0;
    }
    kp.rain_on = h->p.rain_on || h->rain_n > 0 || kp.rframes ? 1 : 0;
    if (h->graph) {
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    return BGF_OK;
}

bgf_status bgf_set_gauges(bgf_handle h, int n, const int* cells, int every) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (n < 0 || n > 16 || (n > 0 && (!cells || every <= 0)))
        return fail(BGF_ERR_INVALID_ARG, "at most 16 gauges, sampled every >= 1 steps");
    int c[16];
    for (int k = 0; k < 16; k++) {
        c[k] = k < n ? cells[k] : -1;
        if (k < n && (c[k] < 0 || (size_t)c[k] >= h->S)) return fail(BGF_ERR_INVALID_ARG, "gauge cell out of range");
    }
    HIPCHK(hipStreamSynchronize(h->stream));
    if (n > 0 && !h->d_gcell) {
        HIPCHK(hipMalloc((void**)&h->d_gcell, sizeof(int) * 16));
        HIPCHK(hipMalloc((void**)&h->d_gring, sizeof(float) * 16 * GAUGE_CAP));
        HIPCHK(hipMalloc((void**)&h->d_gtring, sizeof(double) * GAUGE_CAP));
    }
    if (h->d_gcell) HIPCHK(hipMemcpy(h->d_gcell, c, sizeof(c), hipMemcpyHostToDevice));
    h->gevery = n > 0 ? every : 0;
    h->nstep = 0;
    if (h->graph) {  // the captured period gains (or loses) the sampling launch
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    return BGF_OK;
}

bgf_status bgf_get_gauges(bgf_handle h, float* values, double* times, int* nsamples) {
    if (!h || !nsamples) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    const int ns = h->gevery > 0 ? std::min(h->nstep / h->gevery, GAUGE_CAP) : 0;
    *nsamples = ns;
    if (ns == 0) return BGF_OK;
    if (values) HIPCHK(hipMemcpy(values, h->d_gring, sizeof(float) * 16 * GAUGE_CAP, hipMemcpyDeviceToHost));
    if (times) HIPCHK(hipMemcpy(times, h->d_gtring, sizeof(double) * GAUGE_CAP, hipMemcpyDeviceToHost));
    return BGF_OK;
}

bgf_status bgf_copy_to_host(void* dst, const void* src, size_t n) {
    if ((!dst || !src) && n) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (n) HIPCHK(hipMemcpy(dst, src, n, hipMemcpyDeviceToHost));
    return BGF_OK;
}

bgf_status bgf_refine_flags(bgf_handle h, const char* field, int mode, double a, double b, unsigned char* flags) {
    if (!h || !field || !flags || mode < 0 || mode > 2) return fail(BGF_ERR_INVALID_ARG, "bad argument");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    const std::string f(field);
    const void *x = nullptr, *y = nullptr;
    if (f == "h") x = h->d_h[0];
    else if (f == "u") x = h->d_u[0];
    else if (f == "v") x = h->d_v[0];
    else if (f == "zb") x = h->d_zb;
    else if (f == "zs") { x = h->d_h[0]; y = h->d_zb; }
    else return fail(BGF_ERR_INVALID_ARG, "unknown field " + f);
    if (!h->d_flags) HIPCHK(hipMalloc((void**)&h->d_flags, std::max(h->cap, h->nblkmem)));
    unsigned char* d = h->d_flags;
    HIPCHK(hipMemsetAsync(d, 0, h->nblkmem, h->stream));
    bgf::launch_refine_flags(h->prec, h->kp, x, y, mode, a, b, d, h->stream);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(flags, d, h->nblkmem, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return fail(BGF_ERR_HIP, std::string("refine flags: ") + hipGetErrorString(e));
    return BGF_OK;
}

bgf_status bgf_set_rain_series(bgf_handle h, int n, const double* times, const double* values) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (n != 0 && (n < 2 || !times || !values)) return fail(BGF_ERR_INVALID_ARG, "a rain series needs n >= 2 pairs");
    for (int k = 1; k < n; k++)
        if (!(times[k] > times[k - 1])) return fail(BGF_ERR_INVALID_ARG, "rain series times must increase");
    HIPCHK(hipStreamSynchronize(h->stream));
    (void)hipFree(h->d_rain_t);
    (void)hipFree(h->d_rain_v);
    h->d_rain_t = h->d_rain_v = nullptr;
    h->rain_n = 0;
    if (n > 0) {
        HIPCHK(hipMalloc((void**)&h->d_rain_t, sizeof(double) * n));
        HIPCHK(hipMalloc((void**)&h->d_rain_v, sizeof(double) * n));
        HIPCHK(hipMemcpy(h->d_rain_t, times, sizeof(double) * n, hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(h->d_rain_v, values, sizeof(double) * n, hipMemcpyHostToDevice));
        h->rain_n = n;
    }
    h->kp.rain_on = h->p.rain_on || h->rain_n > 0 || h->kp.rframes ? 1 : 0;
    if (h->graph) {
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    return BGF_OK;
}

bgf_status bgf_set_rain_map(bgf_handle h, int nx, int ny, double xo, double yo, double dx, int nframes, double t0,
                            double dt, const float* frames) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (nframes != 0 && (nx < 2 || ny < 2 || !(dx > 0) || !frames || nframes < 0 || (nframes > 1 && !(dt > 0))))
        return fail(BGF_ERR_INVALID_ARG, "a rain map needs nx, ny >= 2, dx > 0 and dt > 0 between frames");
    HIPCHK(hipStreamSynchronize(h->stream));
    (void)hipFree(h->d_rframes);
    (void)hipFree(h->d_rnow);
    h->d_rframes = h->d_rnow = nullptr;
    bgf::KParams& kp = h->kp;
    kp.rframes = nullptr;
    kp.rnow = nullptr;
    kp.rnframes = 0;
    if (nframes > 0) {
        const size_t n = (size_t)nx * ny;
        HIPCHK(hipMalloc((void**)&h->d_rframes, sizeof(float) * n * nframes));
        HIPCHK(hipMemcpy(h->d_rframes, frames, sizeof(float) * n * nframes, hipMemcpyHostToDevice));
        if (nframes > 1) HIPCHK(hipMalloc((void**)&h->d_rnow, sizeof(float) * n));
        kp.rframes = h->d_rframes;
        kp.rnow = nframes > 1 ? h->d_rnow : h->d_rframes;
        kp.rnx = nx; kp.rny = ny; kp.rnframes = nframes;
        kp.rxo = xo; kp.ryo = yo; kp.rdx = dx; kp.rt0 = t0; kp.rdtf = dt;
    }
    kp.rain_on = h->p.rain_on || h->rain_n > 0 || kp.rframes ? 1 : 0;
    if (h->graph) {
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    return BGF_OK;
}

bgf_status bgf_set_rivers(bgf_handle h, int nriver, const double* boxes, const int* npts, const double* times,
                          const double* flows) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (nriver < 0 || nriver > 64 || (nriver > 0 && (!boxes || !npts || !times || !flows)))
        return fail(BGF_ERR_INVALID_ARG, "0..64 rivers, each with a box and a flow series");
    int tot = 0;
    for (int r = 0; r < nriver; r++) {
        if (npts[r] < 2) return fail(BGF_ERR_INVALID_ARG, "a river flow series needs >= 2 entries");
        for (int k = 1; k < npts[r]; k++)
            if (!(times[tot + k] > times[tot + k - 1])) return fail(BGF_ERR_INVALID_ARG, "river times must increase");
        tot += npts[r];
    }
    HIPCHK(hipStreamSynchronize(h->stream));
    h->riv_box.assign(boxes, boxes + 4 * nriver);
    h->riv_n.assign(npts, npts + nriver);
    h->riv_t.assign(times, times + tot);
    h->riv_q.assign(flows, flows + tot);
    bgf_status s = setup_rivers(h);
    if (h->graph) {
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    return s;
}

namespace {
// A segment's level series on the device (t, then z).
bgf_status upload_series(HostSeg& g) {
    if (g.t.empty()) return BGF_OK;
    const size_t n = g.t.size();
    HIPCHK(hipMalloc((void**)&g.d_series, sizeof(double) * 2 * n));
    HIPCHK(hipMemcpy(g.d_series, g.t.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(g.d_series + n, g.z.data(), sizeof(double) * n, hipMemcpyHostToDevice));
    return BGF_OK;
}

bgf_status check_series(int type, int n, const double* times, const double* levels) {
    if (type < 0 || type > 4) return fail(BGF_ERR_UNSUPPORTED, "boundary types 0 (wall) to 4 are provided");
    if (n != 0 && (n < 2 || !times || !levels)) return fail(BGF_ERR_INVALID_ARG, "a level series needs n >= 2 pairs");
    for (int k = 1; k < n; k++)
        if (!(times[k] > times[k - 1])) return fail(BGF_ERR_INVALID_ARG, "boundary series times must increase");
    return BGF_OK;
}
}  // namespace

bgf_status bgf_set_boundary(bgf_handle h, int side, int type, int n, const double* times, const double* levels) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (side < 0 || side > 3) return fail(BGF_ERR_INVALID_ARG, "side must be 0 (left), 1 (right), 2 (bottom) or 3 (top)");
    if (type < 0 || type > 4) return fail(BGF_ERR_UNSUPPORTED, "boundary types 0 (wall) to 4 are provided");
    if ((type == 2 || type == 3) && (n < 2 || !times || !levels))
        return fail(BGF_ERR_INVALID_ARG, "types 2 and 3 need a water-level series of n >= 2 pairs");
    bgf_status st = check_series(type, type == 2 || type == 3 ? n : 0, times, levels);
    if (st != BGF_OK) return st;
    HIPCHK(hipStreamSynchronize(h->stream));
    HostSeg g;
    g.type = type;
    g.side = side;
    if (type == 2 || type == 3) {
        g.t.assign(times, times + n);
        g.z.assign(levels, levels + n);
    }
    st = upload_series(g);
    if (st != BGF_OK) {
        free_seg(g);
        return st;
    }
    size_t k = 0;
    while (k < h->segs.size() && h->segs[k].side != side) k++;
    if (k < h->segs.size()) {
        free_seg(h->segs[k]);
        h->segs[k] = g;
    } else {
        h->segs.push_back(g);
    }
    return setup_segments(h);
}

bgf_status bgf_set_boundary_segments(bgf_handle h, int nseg, const bgf_bnd_segment* segs) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (nseg < 0 || nseg > BGF_MAX_SEGMENTS || (nseg && !segs))
        return fail(BGF_ERR_INVALID_ARG, "0.." + std::to_string(BGF_MAX_SEGMENTS) + " boundary segments");
    for (int k = 0; k < nseg; k++) {
        const bgf_bnd_segment& g = segs[k];
        if (g.side > 3) return fail(BGF_ERR_INVALID_ARG, "a segment's side is 0..3, or < 0 for its polygon");
        if (g.side < 0 && (g.npoly < 3 || !g.px || !g.py))
            return fail(BGF_ERR_INVALID_ARG, "a segment's polygon needs >= 3 vertices");
        bgf_status st = check_series(g.type, g.nseries, g.times, g.levels);
        if (st != BGF_OK) return st;
    }
    HIPCHK(hipStreamSynchronize(h->stream));
    for (HostSeg& g : h->segs) free_seg(g);
    h->segs.clear();
    for (int k = 0; k < nseg; k++) {
        const bgf_bnd_segment& a = segs[k];
        HostSeg g;
        g.type = a.type;
        g.side = a.side >= 0 ? a.side : -1;
        if (g.side < 0) g.poly = make_polygon(a.npoly, a.px, a.py);
        if (a.nseries > 0) {
            g.t.assign(a.times, a.times + a.nseries);
            g.z.assign(a.levels, a.levels + a.nseries);
        }
        h->segs.push_back(g);
        bgf_status st = upload_series(h->segs.back());
        if (st != BGF_OK) return st;
    }
    return setup_segments(h);
}

bgf_status bgf_set_boundary_map(bgf_handle h, int seg, int nx, int ny, double xo, double yo, double dx, double dy,
                                int nt, double to, double dt, const float* frames) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (seg < 0 || seg >= (int)h->segs.size()) return fail(BGF_ERR_INVALID_ARG, "no boundary segment " + std::to_string(seg));
    if (nx < 2 || ny < 2 || !(dx > 0) || !(dy > 0) || nt < 1 || !frames || (nt > 1 && !(dt > 0)))
        return fail(BGF_ERR_INVALID_ARG, "a level map needs nx, ny >= 2, dx, dy > 0, nt >= 1 frames and dt > 0");
    if ((long long)nx * ny > (1LL << 28)) return fail(BGF_ERR_INVALID_ARG, "a level map holds at most 2^28 values");
    HIPCHK(hipStreamSynchronize(h->stream));
    HostSeg& g = h->segs[seg];
    if (g.d_frames) (void)hipFree(g.d_frames);
    if (g.d_now) (void)hipFree(g.d_now);
    g.d_frames = g.d_now = nullptr;
    g.ext_now = nullptr;
    const size_t n = (size_t)nx * ny;
    std::vector<float> f(frames, frames + n * nt);
    for (float& v : f)
        if (std::isnan(v)) v = 0.0f;  // WLmap.denanval (src/ReadForcing.cu:92)
    HIPCHK(hipMalloc((void**)&g.d_frames, sizeof(float) * f.size()));
    HIPCHK(hipMemcpy(g.d_frames, f.data(), sizeof(float) * f.size(), hipMemcpyHostToDevice));
    if (nt > 1) HIPCHK(hipMalloc((void**)&g.d_now, sizeof(float) * n));
    g.nx = nx; g.ny = ny; g.nt = nt;
    g.xo = xo; g.yo = yo; g.dx = dx; g.dy = dy; g.to = to; g.tdt = nt > 1 ? dt : 1.0;
    return setup_segments(h);
}

bgf_status bgf_set_boundary_map_device(bgf_handle h, int seg, int nx, int ny, double xo, double yo, double dx,
                                       double dy, const float* now_g) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (seg < 0 || seg >= (int)h->segs.size()) return fail(BGF_ERR_INVALID_ARG, "no boundary segment " + std::to_string(seg));
    if (now_g && (nx < 2 || ny < 2 || !(dx > 0) || !(dy > 0)))
        return fail(BGF_ERR_INVALID_ARG, "a level map needs nx, ny >= 2 and dx, dy > 0");
    if (now_g && !device_accessible(now_g)) return fail(BGF_ERR_INVALID_ARG, "now_g is not device memory");
    HIPCHK(hipStreamSynchronize(h->stream));
    HostSeg& g = h->segs[seg];
    if (g.d_frames) (void)hipFree(g.d_frames);
    if (g.d_now) (void)hipFree(g.d_now);
    g.d_frames = g.d_now = nullptr;
    g.ext_now = now_g;
    g.nx = now_g ? nx : 0; g.ny = now_g ? ny : 0; g.nt = 0;
    g.xo = xo; g.yo = yo; g.dx = dx; g.dy = dy; g.to = 0.0; g.tdt = 1.0;
    return setup_segments(h);
}

bgf_status bgf_boundary_blocks(bgf_handle h, int* out) {
    if (!h || !out) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (!h->d_bseg) {  // no segments: every boundary block is the remainder's (index 0)
        for (int k = 0; k < h->nblkmem; k++) out[k] = -1;
        for (int ib : h->active) {
            bool bnd = false;
            for (int k = 0; k < 8; k++) bnd = bnd || h->h_nb[k][ib] == ib;
            if (bnd) out[ib] = 0;
        }
        return BGF_OK;
    }
    std::vector<unsigned char> v(h->nblkmem);
    HIPCHK(hipMemcpy(v.data(), h->d_bseg, v.size(), hipMemcpyDeviceToHost));
    for (int k = 0; k < h->nblkmem; k++) out[k] = v[k] == 255 ? -1 : v[k];
    return BGF_OK;
}

bgf_status bgf_set_boundary_options(bgf_handle h, double zsoffset, double bndtaper, double inittime, double zsinit) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (!std::isfinite(zsoffset) || !std::isfinite(inittime) || !(bndtaper >= 0.0) || std::isinf(zsinit))
        return fail(BGF_ERR_INVALID_ARG, "zsoffset and inittime must be finite, bndtaper >= 0 and zsinit finite or NaN");
    HIPCHK(hipStreamSynchronize(h->stream));
    h->kp.bzsoffset = zsoffset;
    h->kp.btaper = bndtaper;
    h->kp.binittime = inittime;
    h->zsinit = std::isnan(zsinit) ? 0.0 : zsinit;  // FlowbndFlux: zsinit when given, else 0 (src/Boundary.cu:116-120)
    if (h->graph) {  // the captured launches carry the old parameters
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    return setup_segments(h);  // the segments' resting level
}

bgf_status bgf_set_bed_source(bgf_handle h, int nx, int ny, double xo, double yo, double dx, const float* values) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (h->d_bed) {
        HIPCHK(hipStreamSynchronize(h->stream));
        (void)hipFree(h->d_bed);
        h->d_bed = nullptr;
    }
    if (!values) return BGF_OK;
    if (nx < 2 || ny < 2 || !(dx > 0)) return fail(BGF_ERR_INVALID_ARG, "bed source needs nx, ny >= 2 and dx > 0");
    const size_t bytes = sizeof(float) * (size_t)nx * ny;
    HIPCHK(hipMalloc((void**)&h->d_bed, bytes));
    HIPCHK(hipMemcpy(h->d_bed, values, bytes, hipMemcpyHostToDevice));
    h->bed_nx = nx;
    h->bed_ny = ny;
    h->bed_xo = xo;
    h->bed_yo = yo;
    h->bed_dx = dx;
    return BGF_OK;
}

bgf_status bgf_set_stats(bgf_handle h, int mask, double wet_threshold) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (mask < 0 || mask > 7) return fail(BGF_ERR_INVALID_ARG, "statistics mask must be within 0..7");
    HIPCHK(hipStreamSynchronize(h->stream));
    const size_t bytes = h->es * (size_t)h->cap * BS;
    for (int k = 0; k < 15; k++) {
        const int bit = k < 7 ? 1 : k < 14 ? 2 : 4;
        if ((mask & bit) && !h->stats.a[k]) {
            if (hipMalloc(&h->stats.a[k], bytes) != hipSuccess) {
                h->stats.a[k] = nullptr;
                return fail(BGF_ERR_OOM, "statistics allocation failed");
            }
            HIPCHK(hipMemset(h->stats.a[k], 0, bytes));
        } else if (!(mask & bit) && h->stats.a[k]) {
            (void)hipFree(h->stats.a[k]);
            h->stats.a[k] = nullptr;
        }
    }
    h->stats.mask = mask;
    h->stats.wet_threshold = wet_threshold;
    // Initmeanmax (src/Meanmax.cu:191-199): everything reset at the start
    bgf::launch_stats_reset(h->prec == 0 ? 0 : 1, h->kp, h->stats, 7, h->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(h->stream));
    h->stats_n = 0;
    if (h->graph) {  // the captured step gains or loses the statistics kernel
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    return BGF_OK;
}

bgf_status bgf_reset_stats(bgf_handle h, int which) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    bgf::launch_stats_reset(h->prec == 0 ? 0 : 1, h->kp, h->stats, which, h->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipStreamSynchronize(h->stream));
    if (which & 1) h->stats_n = 0;
    return BGF_OK;
}

bgf_status bgf_get_stats(bgf_handle h, const char* name, void* out) {
    if (!h || !name || !out) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    static const char* names[15] = {"hmean", "zsmean", "umean", "vmean", "Umean", "hUmean", "hUUmean", "hmax",
                                    "zsmax", "umax",  "vmax",   "Umax",  "hUmax", "hUUmax", "twet"};
    for (int k = 0; k < 15; k++)
        if (std::strcmp(name, names[k]) == 0) {
            if (!h->stats.a[k]) return fail(BGF_ERR_STATE, std::string(name) + " is not being collected");
            HIPCHK(hipStreamSynchronize(h->stream));
            HIPCHK(hipMemcpy(out, h->stats.a[k], h->es * h->S, hipMemcpyDeviceToHost));
            return BGF_OK;
        }
    return fail(BGF_ERR_INVALID_ARG, std::string("unknown statistic ") + name);
}

bgf_status bgf_sample_raster(bgf_handle h, int nx, int ny, double xo, double yo, double dx, const float* values,
                             void* out) {
    if (!h || !values || !out) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (nx < 2 || ny < 2 || !(dx > 0)) return fail(BGF_ERR_INVALID_ARG, "raster needs nx, ny >= 2 and dx > 0");
    const size_t rbytes = sizeof(float) * (size_t)nx * ny;
    const size_t obytes = h->es * h->S;
    float* d_r = nullptr;
    void* d_o = nullptr;
    HIPCHK(hipMalloc((void**)&d_r, rbytes));
    if (hipMalloc(&d_o, obytes) != hipSuccess) {
        (void)hipFree(d_r);
        return fail(BGF_ERR_OOM, "sample output allocation failed");
    }
    bool ok = hipMemcpy(d_r, values, rbytes, hipMemcpyHostToDevice) == hipSuccess &&
              hipMemcpy(d_o, out, obytes, hipMemcpyHostToDevice) == hipSuccess;
    if (ok) {
        bgf::RemeshLaunch R{};
        R.nblk = h->nblk;
        R.active = h->d_active;
        R.level = h->d_level;
        R.xo = h->d_blkxo;
        R.yo = h->d_blkyo;
        R.nzb = d_o;
        R.bed = d_r;
        R.bnx = nx; R.bny = ny; R.bxo = xo; R.byo = yo; R.bdx = dx;
        R.pxo = h->p.xo; R.pyo = h->p.yo; R.dx = h->p.dx;
        bgf::launch_sample_raster(h->prec == BGF_FP64 ? 0 : 1, R, h->stream);
        ok = hipGetLastError() == hipSuccess && hipStreamSynchronize(h->stream) == hipSuccess &&
             hipMemcpy(out, d_o, obytes, hipMemcpyDeviceToHost) == hipSuccess;
    }
    (void)hipFree(d_r);
    (void)hipFree(d_o);
    if (!ok) return fail(BGF_ERR_HIP, "raster sampling failed");
    return BGF_OK;
}

bgf_status bgf_remesh(bgf_handle h, const bgf_param* p, const bgf_blocks* b, const int* remap) {
    if (!h || !p || !b || !remap) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (!h->state_set) return fail(BGF_ERR_STATE, "state not set");
    // gauge cells are cell indices of the old mesh: a remesh removes the gauges
    h->gevery = 0;
    if (!h->amr)
        return fail(BGF_ERR_UNSUPPORTED, "bgf_remesh needs a multi-level handle (minlevel < maxlevel at bgf_create)");
    bgf_param q = h->p;
    q.nblk = p->nblk;
    q.nblkmem = p->nblkmem;
    const int nbo = h->nblkmem, nbm = q.nblkmem;
    if (q.nblk <= 0 || nbm < q.nblk) return fail(BGF_ERR_INVALID_ARG, "bad sizes");
    MeshInfo mi;
    bgf_status s = check_mesh(&q, b, mi);
    if (s != BGF_OK) return s;
    if (!mi.multilevel) return fail(BGF_ERR_UNSUPPORTED, "an adapted mesh must stay on the multi-level kernels");
    std::vector<char> was(nbo, 0);
    for (int ib : h->active) was[ib] = 1;
    auto old_ok = [&](int i) { return i >= 0 && i < nbo && was[i]; };
    for (int k = 0; k < q.nblk; k++) {
        const int ib = b->active[k];
        const int* r = remap + 5 * ib;
        bool ok = false;
        if (r[0] == 0) ok = r[1] == ib && old_ok(ib);
        else if (r[0] == 1) ok = old_ok(r[1]) && r[2] >= 0 && r[2] < 4;
        else if (r[0] == 2) ok = old_ok(r[1]) && old_ok(r[2]) && old_ok(r[3]) && old_ok(r[4]);
        if (!ok) return fail(BGF_ERR_INVALID_ARG, "remap entry of block " + std::to_string(ib) + " is not valid");
    }
    const int prec = h->prec == 0 ? 0 : 1;
    HIPCHK(hipStreamSynchronize(h->stream));
    if (nbm > h->cap) {
        // grow: a handle with room for twice as many blocks, the state moved into it
        // (a refining run grows a few times at most; each growth re-creates the buffers)
        bgf_handle nh = nullptr;
        s = create_handle(&q, b,
                          (int)std::min<long long>(std::min<long long>(2LL * nbm, kMaxBlocks),
                                                   max_blocks_for(q.precision)),
                          &nh, h);
        if (s != BGF_OK) return s;
        auto undo = [&](bgf_status e) {
            (void)hipStreamSynchronize(nh->stream);
            swap_host_side(nh, h);
            free_handle(nh);
            return e;
        };
        if (hipMemcpy(nh->d_remap, remap, sizeof(int) * 5 * (size_t)nbm, hipMemcpyHostToDevice) != hipSuccess)
            return undo(fail(BGF_ERR_HIP, "remesh: upload failed"));
        bgf::launch_amr_halo(prec, h->kp, h->d_h[0], h->d_u[0], h->d_v[0], h->d_zb, nh->stream);
        bgf::RemeshLaunch R;
        R.nblk = q.nblk;
        R.h = h->d_h[0]; R.u = h->d_u[0]; R.v = h->d_v[0]; R.zb = h->d_zb; R.cf = h->d_cf;
        R.active = nh->d_active; R.level = nh->d_level; R.xo = nh->d_blkxo; R.yo = nh->d_blkyo; R.remap = nh->d_remap;
        R.nh = nh->d_h[0]; R.nu = nh->d_u[0]; R.nv = nh->d_v[0]; R.nzb = nh->d_zb; R.ncf = nh->d_cf;
        R.bed = h->d_bed; R.bnx = h->bed_nx; R.bny = h->bed_ny; R.bxo = h->bed_xo; R.byo = h->bed_yo;
        R.bdx = h->bed_dx; R.pxo = q.xo; R.pyo = q.yo; R.dx = q.dx; R.eps = q.eps;
        bgf::launch_remesh(prec, h->kp, R, nh->stream);
        bgf::launch_amr_fill(prec, nh->kp, nh->d_zb, nh->stream);  // the bed's halo (src/InitialConditions.cu:135-147)
        hipError_t e = hipGetLastError();
        if (e == hipSuccess) e = hipStreamSynchronize(nh->stream);
        if (e != hipSuccess) return undo(fail(BGF_ERR_HIP, std::string("remesh: ") + hipGetErrorString(e)));
        nh->state_set = true;
        nh->timing = h->timing;
        nh->use_graph = h->use_graph;
        std::swap(nh->d_bed, h->d_bed);
        nh->bed_nx = h->bed_nx; nh->bed_ny = h->bed_ny;
        nh->bed_xo = h->bed_xo; nh->bed_yo = h->bed_yo; nh->bed_dx = h->bed_dx;
        std::swap(nh->d_rain_t, h->d_rain_t);
        std::swap(nh->d_rain_v, h->d_rain_v);
        std::swap(nh->d_rframes, h->d_rframes);
        std::swap(nh->d_rnow, h->d_rnow);
        nh->rain_n = h->rain_n;
        const bgf::KParams& ok0 = h->kp;
        nh->kp.rain_on = ok0.rain_on;
        if (ok0.rframes && !h->d_rframes && !nh->d_rframes) {
            // the caller's device map (bgf_set_rain_map_device), read in place
            nh->kp.rframes = ok0.rframes;
            nh->kp.rnow = ok0.rnow;
        } else {
            nh->kp.rframes = nh->d_rframes;
            nh->kp.rnow = ok0.rnow == ok0.rframes ? nh->d_rframes : nh->d_rnow;
        }
        nh->kp.rnx = ok0.rnx; nh->kp.rny = ok0.rny; nh->kp.rnframes = ok0.rnframes;
        nh->kp.rxo = ok0.rxo; nh->kp.ryo = ok0.ryo; nh->kp.rdx = ok0.rdx; nh->kp.rt0 = ok0.rt0; nh->kp.rdtf = ok0.rdtf;
        nh->p.rain_on = h->p.rain_on;
        std::swap(nh->segs, h->segs);  // the boundary segments and their buffers (the table follows the mesh below)
        nh->zsinit = h->zsinit;
        nh->kp.bzsoffset = ok0.bzsoffset;
        nh->kp.btaper = ok0.btaper;
        nh->kp.binittime = ok0.binittime;
        nh->riv_box = h->riv_box; nh->riv_n = h->riv_n; nh->riv_t = h->riv_t; nh->riv_q = h->riv_q;
        std::swap(*h, *nh);  // h takes the new mesh; nh (the old one) is freed
        const int smask = nh->stats.mask;
        const double sthr = nh->stats.wet_threshold;
        free_handle(nh);
        if (smask) {  // the statistics restart on the new mesh
            s = bgf_set_stats(h, smask, sthr);
            if (s != BGF_OK) return s;
        }
        if (!h->riv_n.empty()) {
            s = setup_rivers(h);
            if (s != BGF_OK) return s;
        }
        s = setup_segments(h);  // the boundary blocks of the new mesh
        if (s != BGF_OK) return s;
        g_err.clear();
        return BGF_OK;
    }
    // in place: the new mesh goes to the staging arrays, the new state to the
    // scratch buffers (buffer 1 of h, u, v; two of the stage arrays for the bed
    // and the roughness), then the pointers are exchanged
    const int* src[10] = {b->level, b->LeftBot, b->LeftTop, b->RightBot, b->RightTop,
                          b->TopLeft, b->TopRight, b->BotLeft, b->BotRight, mi.inv.data()};
    bool ok = hipMemcpy(h->d_mesh2[0], b->active, sizeof(int) * q.nblk, hipMemcpyHostToDevice) == hipSuccess;
    for (int k = 0; k < 10; k++)
        ok = ok && hipMemcpy(h->d_mesh2[1 + k], src[k], sizeof(int) * nbm, hipMemcpyHostToDevice) == hipSuccess;
    ok = ok && hipMemcpy(h->d_remap, remap, sizeof(int) * 5 * (size_t)nbm, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(h->d_bxo, b->xo, sizeof(double) * nbm, hipMemcpyHostToDevice) == hipSuccess &&
         hipMemcpy(h->d_byo, b->yo, sizeof(double) * nbm, hipMemcpyHostToDevice) == hipSuccess;
    if (!ok) return fail(BGF_ERR_HIP, "remesh: upload failed");
    bgf::launch_amr_halo(prec, h->kp, h->d_h[0], h->d_u[0], h->d_v[0], h->d_zb, h->stream);
    bgf::RemeshLaunch R;
    R.nblk = q.nblk;
    R.h = h->d_h[0]; R.u = h->d_u[0]; R.v = h->d_v[0]; R.zb = h->d_zb; R.cf = h->d_cf;
    R.active = h->d_mesh2[0]; R.level = h->d_mesh2[1]; R.xo = h->d_bxo; R.yo = h->d_byo; R.remap = h->d_remap;
    R.nh = h->d_h[1]; R.nu = h->d_u[1]; R.nv = h->d_v[1]; R.nzb = h->d_amr[0]; R.ncf = h->d_amr[1];
    R.bed = h->d_bed; R.bnx = h->bed_nx; R.bny = h->bed_ny; R.bxo = h->bed_xo; R.byo = h->bed_yo; R.bdx = h->bed_dx;
    R.pxo = q.xo; R.pyo = q.yo; R.dx = q.dx; R.eps = q.eps;
    bgf::launch_remesh(prec, h->kp, R, h->stream);
    HIPCHK(hipGetLastError());
    std::swap(h->d_h[0], h->d_h[1]);
    std::swap(h->d_u[0], h->d_u[1]);
    std::swap(h->d_v[0], h->d_v[1]);
    std::swap(h->d_zb, h->d_amr[0]);
    std::swap(h->d_cf, h->d_amr[1]);
    std::swap(h->d_active, h->d_mesh2[0]);
    std::swap(h->d_level, h->d_mesh2[1]);
    for (int k = 0; k < 8; k++) std::swap(h->d_nb[k], h->d_mesh2[2 + k]);
    std::swap(h->d_inv, h->d_mesh2[10]);
    std::swap(h->d_blkxo, h->d_bxo);
    std::swap(h->d_blkyo, h->d_byo);
    h->p.nblk = q.nblk;
    h->p.nblkmem = nbm;
    h->nblk = q.nblk;
    h->nblkmem = nbm;
    h->S = (size_t)nbm * BS;
    h->active.assign(b->active, b->active + q.nblk);
    h->xy = block_xy(b, q.nblk, q.dx);
    bgf::KParams& kp = h->kp;
    kp.nblk = q.nblk;
    kp.minlevel = mi.minlev;
    kp.maxlevel = mi.maxlev;
    kp.delta = mi.minlev < 0 ? q.delta * (1 << -mi.minlev) : q.delta / (1 << mi.minlev);
    kp.active = h->d_active;
    kp.level = h->d_level;
    kp.LeftBot = h->d_nb[0]; kp.LeftTop = h->d_nb[1]; kp.RightBot = h->d_nb[2]; kp.RightTop = h->d_nb[3];
    kp.TopLeft = h->d_nb[4]; kp.TopRight = h->d_nb[5]; kp.BotLeft = h->d_nb[6]; kp.BotRight = h->d_nb[7];
    kp.inv = h->d_inv;
    kp.bxo = h->d_blkxo;
    kp.byo = h->d_blkyo;
    bgf::launch_amr_nbr(kp, h->d_nbr, nbm, h->d_rcell, h->d_rmeta, h->stream);
    // the processing order and its block records serve the one-level kernels only,
    // which a multi-level handle never runs: they are not rebuilt here
    ok = hipGetLastError() == hipSuccess;
    if (q.spherical) ok = ok && upload_metric(h, &q, b, nbm);
    if (!ok) return fail(BGF_ERR_HIP, "remesh: upload failed");
    kp.grid_pred = bgf::persistent_grid(h->prec, 0, q.nblk, h->wg_pred);
    kp.grid_corr = bgf::persistent_grid(h->prec, 1, q.nblk, h->wg_corr);
    h->h_level.assign(b->level, b->level + nbm);
    h->h_xo.assign(b->xo, b->xo + nbm);
    h->h_yo.assign(b->yo, b->yo + nbm);
    {
        const int* nb[8] = {b->LeftBot, b->LeftTop, b->RightBot, b->RightTop, b->TopLeft, b->TopRight, b->BotLeft, b->BotRight};
        for (int k = 0; k < 8; k++) h->h_nb[k].assign(nb[k], nb[k] + nbm);
    }
    if (!h->segs.empty()) {
        HIPCHK(hipStreamSynchronize(h->stream));
        s = setup_segments(h);  // the boundary blocks of the new mesh
    } else {
        s = setup_fix(h);
    }
    if (s != BGF_OK) return s;
    if (!h->riv_n.empty()) {
        HIPCHK(hipStreamSynchronize(h->stream));
        s = setup_rivers(h);  // the discharge cells of the new mesh
        if (s != BGF_OK) return s;
    }
    // the bed's halo on the new mesh (src/InitialConditions.cu:135-147)
    bgf::launch_amr_fill(prec, kp, h->d_zb, h->stream);
    // the statistics restart on the new mesh
    bgf::launch_stats_reset(prec, kp, h->stats, 7, h->stream);
    h->stats_n = 0;
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return fail(BGF_ERR_HIP, std::string("remesh: ") + hipGetErrorString(e));
    if (h->graph) {
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    g_err.clear();
    return BGF_OK;
}

bgf_status bgf_last_run_steps(bgf_handle h, int* nsteps) {
    if (!h || !nsteps) return fail(BGF_ERR_INVALID_ARG, "null argument");
    *nsteps = h->last_steps;
    return BGF_OK;
}

bgf_status bgf_volume(bgf_handle h, double* volume) {
    if (!h || !volume) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    bgf::launch_volume(h->prec, h->kp, h->d_h[0], h->d_volpart, h->d_volout, h->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(volume, h->d_volout, sizeof(double), hipMemcpyDeviceToHost, h->stream));
    HIPCHK(hipStreamSynchronize(h->stream));
    return BGF_OK;
}

bgf_status bgf_device_array(bgf_handle h, const char* name, void** devptr) {
    if (!h || !name || !devptr) return fail(BGF_ERR_INVALID_ARG, "null argument");
    std::string n(name);
    void* p = nullptr;
    if (n == "h") p = h->d_h[0];
    else if (n == "u") p = h->d_u[0];
    else if (n == "v") p = h->d_v[0];
    else if (n == "ho") p = h->d_h[1];
    else if (n == "uo") p = h->d_u[1];
    else if (n == "vo") p = h->d_v[1];
    else if (n == "zb") p = h->d_zb;
    else if (n == "cf") {
        p = h->d_cf;
        h->cf_shared = true;  // the caller may write it: read it per cell from now on
        if (h->kp.cf_uniform) {
            h->kp.cf_uniform = 0;
            if (h->graph) {
                (void)hipGraphExecDestroy(h->graph);
                h->graph = nullptr;
            }
        }
    }
    else if (n == "dh") p = h->d_dh;
    else if (n == "dhu") p = h->d_dhu;
    else if (n == "dhv") p = h->d_dhv;
    else return fail(BGF_ERR_INVALID_ARG, "unknown array " + n);
    *devptr = p;
    return BGF_OK;
}

bgf_status bgf_set_schedule(bgf_handle h, int tile_x, int tile_y, int wg_pred, int wg_corr) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (h->pending_steps) return fail(BGF_ERR_STATE, "bgf_run_async pending: call bgf_sync first");
    if (tile_x < 0 || tile_y < 0 || tile_x > 4096 || tile_y > 4096 || wg_pred < 0 || wg_corr < 0 || wg_pred > 64 ||
        wg_corr > 64)
        return fail(BGF_ERR_INVALID_ARG, "schedule out of range");
    const int tx = tile_x ? tile_x : h->tile_x, ty = tile_y ? tile_y : h->tile_y;
    if (tx != h->tile_x || ty != h->tile_y) {
        if (!h->amr) {  // multi-level meshes have no processing order
            std::vector<int> order = processing_order(h->xy, tx, ty);
            HIPCHK(hipStreamSynchronize(h->stream));
            HIPCHK(hipMemcpy(h->d_order, order.data(), sizeof(int) * h->nblk, hipMemcpyHostToDevice));
            bgf::launch_records(h->kp, h->d_rec, h->stream);
            HIPCHK(hipGetLastError());
        }
        h->tile_x = tx;
        h->tile_y = ty;
    }
    const int gp = bgf::persistent_grid(h->prec, 0, h->nblk, wg_pred);
    const int gc = bgf::persistent_grid(h->prec, 1, h->nblk, wg_corr);
    if (gp <= 0 || gc <= 0) return fail(BGF_ERR_HIP, "occupancy query failed");
    h->wg_pred = wg_pred;
    h->wg_corr = wg_corr;
    h->kp.grid_pred = gp;
    h->kp.grid_corr = gc;
    if (h->graph) {
        (void)hipGraphExecDestroy(h->graph);
        h->graph = nullptr;
    }
    g_err.clear();
    return BGF_OK;
}

bgf_status bgf_get_schedule(bgf_handle h, int* tile_x, int* tile_y, int* wg_pred, int* wg_corr, int* grid_pred,
                            int* grid_corr) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    if (tile_x) *tile_x = h->tile_x;
    if (tile_y) *tile_y = h->tile_y;
    if (wg_pred) *wg_pred = h->wg_pred;
    if (wg_corr) *wg_corr = h->wg_corr;
    if (grid_pred) *grid_pred = h->kp.grid_pred;
    if (grid_corr) *grid_corr = h->kp.grid_corr;
    return BGF_OK;
}

bgf_status bgf_set_timing(bgf_handle h, int enable) {
    if (!h) return fail(BGF_ERR_INVALID_ARG, "null handle");
    h->timing = enable != 0;
    h->t_pred = h->t_red = h->t_corr = 0;
    h->t_n = 0;
    return BGF_OK;
}

bgf_status bgf_kernel_times(bgf_handle h, int n, const char** names, double* ms, int* count) {
    if (!h || !count) return fail(BGF_ERR_INVALID_ARG, "null argument");
    static const char* kn[3] = {"k_predictor", "k_reduce_dt", "k_corrector"};
    double v[3] = {h->t_pred, h->t_red, h->t_corr};
    int c = 0;
    for (int k = 0; k < 3 && k < n; k++) {
        if (names) names[k] = kn[k];
        if (ms) ms[k] = h->t_n ? v[k] / h->t_n : 0.0;
        c++;
    }
    *count = c;
    return BGF_OK;
}

// Uniform block list with the raster order of InitBlockxoyo and the
// neighbour convention of InitBlockneighbours (src/Mesh.cu:257-433): block
// (bx, by) is number by*nbx + bx and a missing neighbour is the block itself.
bgf_status bgf_mesh_uniform(int nbx, int nby, double dx, int level, int dbl, int* active, int* lev, double* xo,
                            double* yo, int* LeftBot, int* LeftTop, int* RightBot, int* RightTop, int* TopLeft,
                            int* TopRight, int* BotLeft, int* BotRight) {
    if (nbx <= 0 || nby <= 0 || !active || !lev || !xo || !yo) return fail(BGF_ERR_INVALID_ARG, "bad mesh arguments");
    double levdx = level < 0 ? dx * (1 << -level) : dx / (1 << level);
    for (int by = 0; by < nby; by++)
        for (int bx = 0; bx < nbx; bx++) {
            int ib = by * nbx + bx;
            active[ib] = ib;
            lev[ib] = level;
            if (dbl) {
                xo[ib] = bx * ((double)BW) * levdx + 0.5 * levdx;
                yo[ib] = by * ((double)BW) * levdx + 0.5 * levdx;
            } else {
                xo[ib] = (double)(bx * ((float)BW) * (float)levdx + 0.5f * (float)levdx);
                yo[ib] = (double)(by * ((float)BW) * (float)levdx + 0.5f * (float)levdx);
            }
            int l = bx > 0 ? ib - 1 : ib, r = bx < nbx - 1 ? ib + 1 : ib;
            int bt = by > 0 ? ib - nbx : ib, t = by < nby - 1 ? ib + nbx : ib;
            LeftBot[ib] = LeftTop[ib] = l;
            RightBot[ib] = RightTop[ib] = r;
            BotLeft[ib] = BotRight[ib] = bt;
            TopLeft[ib] = TopRight[ib] = t;
        }
    return BGF_OK;
}

// Block list of a quadtree mesh given by its leaves.  Leaf k is block k, at
// level lev[k] with integer position (ix[k], iy[k]) among the blocks of that
// level; the domain is nbx x nby blocks of level `base`.  Neighbours follow
// the convention of the reference's adaptation (src/Adaptation.cu:1017-1795):
// a side shared with one block of the same or a coarser level points both
// halves at it, a side shared with two finer blocks points the first half
// (bottom or left) and the second half at them, and a side on the domain
// edge points at the block itself.  The leaves must tile the domain exactly
// and neighbouring levels may differ by one at most.
bgf_status bgf_mesh_from_leaves(int nleaf, const int* lev, const int* ix, const int* iy, int nbx, int nby, int base,
                                double dx, int* active, int* level, double* xo, double* yo, int* LeftBot,
                                int* LeftTop, int* RightBot, int* RightTop, int* TopLeft, int* TopRight,
                                int* BotLeft, int* BotRight) {
    if (nleaf <= 0 || nbx <= 0 || nby <= 0 || !lev || !ix || !iy || !active || !level || !xo || !yo)
        return fail(BGF_ERR_INVALID_ARG, "bad mesh arguments");
    std::vector<int> id(nleaf);
    std::vector<long long> x(nleaf), y(nleaf);
    for (int k = 0; k < nleaf; k++) {
        id[k] = k;
        x[k] = ix[k];
        y[k] = iy[k];
    }
    bgf_status s = quadtree_neighbours(nleaf, id.data(), lev, x.data(), y.data(), nbx, nby, base, LeftBot, LeftTop,
                                       RightBot, RightTop, TopLeft, TopRight, BotLeft, BotRight);
    if (s != BGF_OK) return s;
    for (int k = 0; k < nleaf; k++) {
        active[k] = k;
        level[k] = lev[k];
        const double ldx = level_dx(dx, lev[k]);
        xo[k] = ix[k] * (double)BW * ldx + 0.5 * ldx;
        yo[k] = iy[k] * (double)BW * ldx + 0.5 * ldx;
    }
    return BGF_OK;
}

}  // extern "C"
