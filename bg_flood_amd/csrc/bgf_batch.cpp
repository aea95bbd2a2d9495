// bgf_batch.cpp -- batches of independent one-level domains (ensembles and
// continuous batching of solve requests) advanced by one set of launches.
//
// The members' blocks are packed into one block list of fixed capacity: a
// member owns a contiguous range of block slots (its own nblkmem blocks, with
// neighbour indices offset into the range), so one predictor / reduction /
// corrector launch advances every member.  Each member keeps its own loop
// state (time step, time, end time, rain rate) in one DevLoop: the predictor
// merges block minima into the member's slots, the reduction runs one wave per
// member, and the corrector reads the member's dt.  Members that reached their
// end time are skipped, members can be added and removed between runs, and
// their states stay resident in HBM.  The reference has no counterpart: it
// runs one domain per process (src/Mainloop.cu:17-91).
//
// A batch whose common parameters span several levels (maxlevel > minlevel)
// holds multi-level domains instead and steps them with the multi-level
// kernels: one set of launches covers every member's blocks, each block
// finds its member's loop state through the block-to-member table, and the
// blocks of one member keep their relative order in the packed active list,
// which the wet/dry prolongation's sequential semantics rest on.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <vector>

#include "bgf_host.h"

using namespace bgf_host;

namespace {

struct Member {
    bool used = false;
    int off = 0;      // first block slot of the member's range
    int nblk = 0;     // active blocks
    int nblkmem = 0;  // block slots
    std::vector<int> active;  // global block ids, in the member's own active order
    std::vector<int> order;   // global block ids, tiled processing order
    std::vector<int> fix;     // multi-level: global ids of the blocks that wait for others' faces
    bool fix_all = false, odd = false;
    BlockXY xy;               // block coordinates (global ids), for re-tiling
    double rain = 0.0;
    std::vector<int> gauges;  // global cell indices
};

}  // namespace

struct bgf_batch_s {
    bgf_param common;
    int prec = 0;
    size_t es = 4;
    int cap_blocks = 0, cap_members = 0;
    size_t S = 0;
    std::vector<Member> members;
    std::vector<int> slot_owner;  // member of each block slot, -1 if free
    std::vector<bgf::DevLoop> loops;  // host mirror of the device loop states
    int *d_active = nullptr, *d_order = nullptr, *d_sid = nullptr, *d_level = nullptr;
    int* d_queue = nullptr;  // work-queue counters of the persistent kernels
    int* d_rec = nullptr;    // per-position block records of the processing order
    int* d_nb[8] = {nullptr};
    void *d_h[2] = {nullptr, nullptr}, *d_u[2] = {nullptr, nullptr}, *d_v[2] = {nullptr, nullptr};
    void *d_zb = nullptr, *d_cf = nullptr, *d_dh = nullptr, *d_dhu = nullptr, *d_dhv = nullptr, *d_hmax = nullptr;
    void* d_ch = nullptr;  // compensation of h (BGF_FP32_COMP)
    double *d_volpart = nullptr, *d_volout = nullptr;
    int* d_gcell = nullptr;    // gauge cells, 16 per member slot
    float* d_gval = nullptr;   // sampled depths
    float* d_ring = nullptr;   // per-step gauge series: NSAMP samples of 16 gauges per member slot
    double* d_tring = nullptr; // their times
    bool gauges_on = false;    // some member records gauge series
    bool track_max = false;    // the corrector folds every step's depth into hmax
    bgf::DevLoop* d_loop = nullptr;
    bgf::KParams kp;
    hipStream_t stream = nullptr;
    int pending = 0;
    long long cell_updates = 0;
    int nactive_blocks = 0;
    int wg_pred = 0, wg_corr = 0;
    int tile_x = TILE_X, tile_y = TILE_Y;
    bool use_graph = true;
    hipGraphExec_t graph = nullptr;  // PERIOD batch steps; rebuilt after membership changes
    // multi-level members: position of each block slot in the packed active
    // list, the neighbour records, and the gradient / face / snapshot arrays
    bool amr = false;
    int* d_inv = nullptr;
    int* d_nbr = nullptr;
    int4* d_rcell = nullptr;  // with d_rmeta and d_fix behind it
    int2* d_rmeta = nullptr;
    int* d_fix = nullptr;
    void* d_amr[11] = {nullptr};  // as a handle's: 2-9 face fluxes, 10 hsnap (0-1, remesh staging, unused)
    // the persistent kernels walk only the blocks of members still running:
    // their processing order, launch parameters, and the members it was built for
    bgf::KParams krun;
    std::vector<int> run_members;
    bool run_valid = false;
    std::unique_ptr<ReadBack> back{new ReadBack};
};

namespace {

// Steps of a captured graph, as a handle's: even, and used by runs of twice as many and more.
constexpr int PERIOD = 8;
constexpr int NGAUGE = 16;
constexpr int NSAMP = 2048;  // gauge samples kept per member

void free_batch(bgf_batch b) {
    auto F = [](void* p) { if (p) (void)hipFree(p); };
    F(b->d_active); F(b->d_order); F(b->d_sid); F(b->d_level); F(b->d_queue); F(b->d_rec);
    for (int k = 0; k < 8; k++) F(b->d_nb[k]);
    for (int k = 0; k < 2; k++) { F(b->d_h[k]); F(b->d_u[k]); F(b->d_v[k]); }
    F(b->d_zb); F(b->d_cf); F(b->d_dh); F(b->d_dhu); F(b->d_dhv); F(b->d_hmax); F(b->d_ch);
    F(b->d_volpart); F(b->d_volout); F(b->d_gcell); F(b->d_gval); F(b->d_loop);
    F(b->d_ring); F(b->d_tring);
    F(b->d_inv); F(b->d_nbr); F(b->d_rcell);
    for (int k = 0; k < 11; k++) F(b->d_amr[k]);
    if (b->graph) (void)hipGraphExecDestroy(b->graph);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
}

bgf::DevLoop empty_loop() {
    bgf::DevLoop L;
    std::memset(&L, 0, sizeof(L));
    L.done = 1;
    for (int k = 0; k < bgf::NSLOT; k++) {
        L.slot32[k] = 0x7f800000u;
        L.slot64[k] = 0x7ff0000000000000ull;
    }
    return L;
}

// Rebuilds the packed active list, processing order and member ids after a
// membership change, and the launch parameters that depend on them.
bgf_status rebuild(bgf_batch b) {
    std::vector<int> active, order, sid(b->cap_blocks, 0);
    for (int m = 0; m < b->cap_members; m++) {
        const Member& M = b->members[m];
        if (!M.used) continue;
        active.insert(active.end(), M.active.begin(), M.active.end());
        order.insert(order.end(), M.order.begin(), M.order.end());
        for (int k = 0; k < M.nblkmem; k++) sid[M.off + k] = m;
    }
    b->nactive_blocks = (int)active.size();
    b->run_valid = false;
    if (b->graph) {
        (void)hipGraphExecDestroy(b->graph);
        b->graph = nullptr;
    }
    if (!active.empty()) {
        HIPCHK(hipMemcpy(b->d_active, active.data(), sizeof(int) * active.size(), hipMemcpyHostToDevice));
        HIPCHK(hipMemcpy(b->d_order, order.data(), sizeof(int) * order.size(), hipMemcpyHostToDevice));
    }
    HIPCHK(hipMemcpy(b->d_sid, sid.data(), sizeof(int) * sid.size(), hipMemcpyHostToDevice));
    b->kp.nblk = b->nactive_blocks;
    if (b->amr) {
        std::vector<int> inv(b->cap_blocks, -1);
        for (size_t k = 0; k < active.size(); k++) inv[active[k]] = (int)k;
        HIPCHK(hipMemcpy(b->d_inv, inv.data(), sizeof(int) * inv.size(), hipMemcpyHostToDevice));
        bgf::launch_amr_nbr(b->kp, b->d_nbr, b->cap_blocks, b->d_rcell, b->d_rmeta, b->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(b->stream));
    }
    return BGF_OK;
}

// Processing order over the members that have not reached their end time,
// rebuilt when that set changes (finished members cost nothing afterwards).
bgf_status prepare_run(bgf_batch b) {
    std::vector<int> running;
    for (int m = 0; m < b->cap_members; m++)
        if (b->members[m].used && !b->loops[m].done) running.push_back(m);
    if (b->run_valid && running == b->run_members) return BGF_OK;
    std::vector<int> order;
    for (int m : running) order.insert(order.end(), b->members[m].order.begin(), b->members[m].order.end());
    if (!order.empty())
        HIPCHK(hipMemcpy(b->d_order, order.data(), sizeof(int) * order.size(), hipMemcpyHostToDevice));
    b->krun = b->kp;
    b->krun.nblk = (int)order.size();
    b->krun.hmax = b->track_max ? (float*)b->d_hmax : nullptr;
    if (b->amr) {
        b->krun.active = b->d_order;  // the multi-level kernels walk the running members' active lists
        bool all = false, odd = false;
        for (int m : running) {
            all = all || b->members[m].fix_all;
            odd = odd || b->members[m].odd;
        }
        std::vector<int> fix = all ? order : std::vector<int>();
        for (int m : running)
            if (!all) fix.insert(fix.end(), b->members[m].fix.begin(), b->members[m].fix.end());
        if (!fix.empty())
            HIPCHK(hipMemcpy(b->d_fix, fix.data(), sizeof(int) * fix.size(), hipMemcpyHostToDevice));
        b->krun.fix = b->d_fix;
        b->krun.nfix = (int)fix.size();
        b->krun.fix_all = all ? 1 : 0;
        b->krun.odd = odd ? 1 : 0;
    }
    if (!order.empty() && !b->amr) {
        b->krun.grid_pred = bgf::persistent_grid(b->prec, 0, b->krun.nblk, b->wg_pred);
        b->krun.grid_corr = bgf::persistent_grid(b->prec, 1, b->krun.nblk, b->wg_corr);
        if (b->krun.grid_pred <= 0 || b->krun.grid_corr <= 0) return fail(BGF_ERR_HIP, "occupancy query failed");
        bgf::launch_records(b->krun, b->d_rec, b->stream);
        HIPCHK(hipGetLastError());
    }
    b->run_members = running;
    b->run_valid = true;
    if (b->graph) {
        (void)hipGraphExecDestroy(b->graph);
        b->graph = nullptr;
    }
    return BGF_OK;
}

// Launch parameters restricted to one member's blocks.
bgf::KParams member_view(bgf_batch b, int m, int aoff) {
    bgf::KParams P = b->kp;
    P.active = b->d_active + aoff;
    P.nblk = b->members[m].nblk;
    return P;
}

int active_offset(bgf_batch b, int m) {
    int a = 0;
    for (int k = 0; k < m; k++)
        if (b->members[k].used) a += b->members[k].nblk;
    return a;
}

bgf_status check_member(bgf_batch b, int m) {
    if (!b) return fail(BGF_ERR_INVALID_ARG, "null batch");
    if (m < 0 || m >= b->cap_members || !b->members[m].used) return fail(BGF_ERR_INVALID_ARG, "no such member");
    if (b->pending) return fail(BGF_ERR_STATE, "bgf_batch_run_async pending: call bgf_batch_sync first");
    return BGF_OK;
}

// Enqueues nsteps batch steps starting at buffer parity 0.
template <class T> void fill_amr(bgf_batch b, bgf::AmrBuffers<T>* B) {
    B->h = (T*)b->d_h[0]; B->u = (T*)b->d_u[0]; B->v = (T*)b->d_v[0];
    B->ho = (T*)b->d_h[1]; B->uo = (T*)b->d_u[1]; B->vo = (T*)b->d_v[1];
    B->zb = (T*)b->d_zb; B->cf = (const T*)b->d_cf;
    T** f[8] = {&B->Fhu, &B->Fqux, &B->Su, &B->Fqvx, &B->Fhv, &B->Fqvy, &B->Sv, &B->Fquy};
    for (int k = 0; k < 8; k++) *f[k] = (T*)b->d_amr[2 + k];
    B->hsnap = (T*)b->d_amr[10];
    B->dh = (T*)b->d_dh; B->dhu = (T*)b->d_dhu; B->dhv = (T*)b->d_dhv;
}

void enqueue_steps(bgf_batch b, int nsteps) {
    alignas(16) unsigned char storage[sizeof(bgf::AmrBuffers<double>) > sizeof(bgf::StepBuffers<double>)
                                          ? sizeof(bgf::AmrBuffers<double>)
                                          : sizeof(bgf::StepBuffers<double>)];
    if (b->amr) {
        // the state stays in buffer 0; buffer 1 holds the predictor's stage
        if (b->prec == 0) fill_amr(b, (bgf::AmrBuffers<double>*)storage);
        else fill_amr(b, (bgf::AmrBuffers<float>*)storage);
        for (int k = 0; k < nsteps; k++) {
            bgf::launch_amr_step(b->prec, b->krun, storage, b->d_loop, nullptr, 1, b->stream, nullptr);
            if (b->gauges_on)
                bgf::launch_gauge_step(b->prec, b->d_h[0], b->d_gcell, b->d_loop, b->cap_members, NSAMP, b->d_ring,
                                       b->d_tring, b->stream);
        }
        return;
    }
    for (int k = 0; k < nsteps; k++) {
        const int in = k & 1, out = 1 - in;
        if (b->prec == 0) {
            auto* B = (bgf::StepBuffers<double>*)storage;
            *B = {(const double*)b->d_h[in], (const double*)b->d_u[in], (const double*)b->d_v[in],
                  (double*)b->d_h[out], (double*)b->d_u[out], (double*)b->d_v[out], (const double*)b->d_zb,
                  (const double*)b->d_cf, (double*)b->d_dh, (double*)b->d_dhu, (double*)b->d_dhv, nullptr};
        } else {
            auto* B = (bgf::StepBuffers<float>*)storage;
            *B = {(const float*)b->d_h[in], (const float*)b->d_u[in], (const float*)b->d_v[in],
                  (float*)b->d_h[out], (float*)b->d_u[out], (float*)b->d_v[out], (const float*)b->d_zb,
                  (const float*)b->d_cf, (float*)b->d_dh, (float*)b->d_dhu, (float*)b->d_dhv, (float*)b->d_ch};
        }
        bgf::launch_step(b->prec, b->krun, storage, b->d_loop, nullptr, 1, b->stream, nullptr);
        if (b->gauges_on)
            bgf::launch_gauge_step(b->prec, b->d_h[out], b->d_gcell, b->d_loop, b->cap_members, NSAMP, b->d_ring,
                                   b->d_tring, b->stream);
    }
}

}  // namespace

extern "C" {

bgf_status bgf_batch_create(const bgf_param* common, int max_blocks, int max_members, bgf_batch* out) {
    if (!out || max_blocks <= 0 || max_members <= 0) return fail(BGF_ERR_INVALID_ARG, "bad batch arguments");
    if (max_blocks > kMaxBlocks)
        return fail(BGF_ERR_UNSUPPORTED, "max_blocks above " + std::to_string(kMaxBlocks) +
                                             ": cell indices would not fit in 32 bits");
    if (common && !block_bytes_ok(max_blocks, common->precision))
        return fail(BGF_ERR_UNSUPPORTED, "max_blocks above the 32-bit byte offset limit of this precision");
    *out = nullptr;
    bgf_param p = *common;
    p.nblk = 1;
    p.nblkmem = 1;
    bgf_status s = check_param(&p);
    if (s != BGF_OK) return s;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(BGF_ERR_NO_DEVICE, "no HIP device");
    auto* b = new bgf_batch_s();
    // BGF_GRAPH=0 launches every step's kernels directly instead of replaying a captured graph
    if (const char* e = std::getenv("BGF_GRAPH")) b->use_graph = std::atoi(e) != 0;
    b->common = *common;
    b->prec = common->precision;
    b->es = b->prec == 0 ? sizeof(double) : sizeof(float);
    b->cap_blocks = max_blocks;
    b->cap_members = max_members;
    b->S = (size_t)max_blocks * BS;
    b->members.assign(max_members, Member());
    b->slot_owner.assign(max_blocks, -1);
    b->loops.assign(max_members, empty_loop());
    auto A = [&](void** ptr, size_t bytes) -> bool {
        if (hipMalloc(ptr, bytes) != hipSuccess) return false;
        return hipMemset(*ptr, 0, bytes) == hipSuccess;
    };
    bool ok = A((void**)&b->d_active, sizeof(int) * max_blocks) && A((void**)&b->d_order, sizeof(int) * max_blocks) &&
              A((void**)&b->d_sid, sizeof(int) * max_blocks) && A((void**)&b->d_level, sizeof(int) * max_blocks) &&
              A((void**)&b->d_queue, sizeof(int) * 2 * bgf::NXCD * bgf::QSTRIDE) &&
              A((void**)&b->d_rec, sizeof(int) * 8 * (size_t)max_blocks);
    for (int k = 0; k < 8; k++) ok = ok && A((void**)&b->d_nb[k], sizeof(int) * max_blocks);
    for (int k = 0; k < 2; k++)
        ok = ok && A(&b->d_h[k], b->es * b->S) && A(&b->d_u[k], b->es * b->S) && A(&b->d_v[k], b->es * b->S);
    ok = ok && A(&b->d_zb, b->es * b->S) && A(&b->d_cf, b->es * b->S) && A(&b->d_dh, b->es * b->S) &&
         A(&b->d_dhu, b->es * b->S) && A(&b->d_dhv, b->es * b->S) && A(&b->d_hmax, sizeof(float) * b->S);
    ok = ok && A((void**)&b->d_volpart, sizeof(double) * max_blocks) && A((void**)&b->d_volout, sizeof(double));
    if (b->prec == BGF_FP32_COMP) ok = ok && A(&b->d_ch, b->es * b->S);
    ok = ok && A((void**)&b->d_gcell, sizeof(int) * NGAUGE * max_members) &&
         A((void**)&b->d_gval, sizeof(float) * NGAUGE * max_members);
    ok = ok && A((void**)&b->d_loop, sizeof(bgf::DevLoop) * max_members);
    ok = ok && hipMemset(b->d_gcell, 0xff, sizeof(int) * NGAUGE * max_members) == hipSuccess;  // no gauges: -1
    ok = ok && A((void**)&b->d_ring, sizeof(float) * NGAUGE * NSAMP * max_members) &&
         A((void**)&b->d_tring, sizeof(double) * NSAMP * max_members);
    b->amr = common->maxlevel > common->minlevel;
    if (b->amr) {
        ok = ok && A((void**)&b->d_inv, sizeof(int) * max_blocks) && A((void**)&b->d_nbr, sizeof(int) * bgf::NBR * (size_t)max_blocks) &&
             mesh_tables((size_t)max_blocks, &b->d_rcell, &b->d_rmeta, &b->d_fix);
        for (int k = 2; k < 11; k++) ok = ok && A(&b->d_amr[k], b->es * b->S);
    }
    if (!ok) {
        free_batch(b);
        (void)hipGetLastError();
        return fail(BGF_ERR_OOM, "device allocation failed");
    }
    if (hipStreamCreate(&b->stream) != hipSuccess) {
        free_batch(b);
        return fail(BGF_ERR_HIP, "stream creation failed");
    }
    bgf::KParams& kp = b->kp;
    kp.g = p.g; kp.eps = p.eps; kp.CFL = p.CFL; kp.theta = p.theta;
    kp.delta0 = p.delta;
    kp.delta = p.delta;  // one-level members are grids of level 0 (checked at add)
    kp.minlevel = b->amr ? common->minlevel : 0;
    kp.maxlevel = b->amr ? common->maxlevel : 0;
    kp.inv = b->d_inv;
    kp.nbr = b->d_nbr;
    kp.rcell = b->d_rcell;
    kp.rmeta = b->d_rmeta;
    kp.fc = p.precision == 0 ? coriolis<double>(p.lat) : coriolis<float>(p.lat);
    kp.mask = p.mask;
    kp.frictionmodel = p.frictionmodel;
    kp.aoibnd = p.aoibnd;
    kp.ForceMassConserve = p.ForceMassConserve;
    kp.rain_on = p.rain_on;
    kp.wetdryfix = p.wetdryfix;
    kp.active = b->d_active;
    kp.order = b->d_order;
    kp.rec = b->d_rec;
    kp.queue = b->d_queue;
    kp.LeftBot = b->d_nb[0]; kp.LeftTop = b->d_nb[1]; kp.RightBot = b->d_nb[2]; kp.RightTop = b->d_nb[3];
    kp.TopLeft = b->d_nb[4]; kp.TopRight = b->d_nb[5]; kp.BotLeft = b->d_nb[6]; kp.BotRight = b->d_nb[7];
    kp.level = b->d_level;
    kp.sid = b->d_sid;
    kp.nmember = max_members;
    if (const char* e = std::getenv("BGF_WG_PER_CU")) std::sscanf(e, "%d,%d", &b->wg_pred, &b->wg_corr);
    std::vector<bgf::DevLoop> L(max_members, empty_loop());
    if (hipMemcpy(b->d_loop, L.data(), sizeof(bgf::DevLoop) * max_members, hipMemcpyHostToDevice) != hipSuccess) {
        free_batch(b);
        return fail(BGF_ERR_HIP, "loop upload failed");
    }
    *out = b;
    g_err.clear();
    return BGF_OK;
}

bgf_status bgf_batch_destroy(bgf_batch b) {
    if (!b) return fail(BGF_ERR_INVALID_ARG, "null batch");
    (void)hipStreamSynchronize(b->stream);
    free_batch(b);
    return BGF_OK;
}

bgf_status bgf_batch_add(bgf_batch b, const bgf_param* p, const bgf_blocks* blk, const void* zb, const void* hh,
                         const void* u, const void* v, const void* cf, double dtinit, double endtime, int* member) {
    if (!b || !p || !blk || !zb || !hh || !u || !v || !cf || !member) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (b->pending) return fail(BGF_ERR_STATE, "bgf_batch_run_async pending: call bgf_batch_sync first");
    bgf_status s = check_param(p);
    if (s != BGF_OK) return s;
    if (p->spherical) return fail(BGF_ERR_UNSUPPORTED, "batch members must be Cartesian grids");
    const bgf_param& c = b->common;
    if (p->precision != c.precision || p->g != c.g || p->eps != c.eps || p->CFL != c.CFL || p->theta != c.theta ||
        p->delta != c.delta || p->frictionmodel != c.frictionmodel || p->aoibnd != c.aoibnd ||
        p->ForceMassConserve != c.ForceMassConserve || p->lat != c.lat || p->mask != c.mask || p->rain_on != c.rain_on)
        return fail(BGF_ERR_INVALID_ARG, "member parameters must match the batch's except nblk, nblkmem and rain");
    const int nblk = p->nblk, nbm = p->nblkmem;
    std::vector<int> seen(nbm, 0);
    for (int k = 0; k < nblk; k++) {
        const int ib = blk->active[k];
        if (ib < 0 || ib >= nbm || seen[ib]++) return fail(BGF_ERR_INVALID_ARG, "bad active list");
    }
    if (b->amr) {
        // multi-level members: levels within the batch's range, neighbours among the member's blocks
        if (p->minlevel < c.minlevel || p->maxlevel > c.maxlevel || p->dx != c.dx || p->wetdryfix != c.wetdryfix)
            return fail(BGF_ERR_INVALID_ARG, "member levels outside the batch's, or a different dx or wetdryfix");
        const int* nbs[8] = {blk->LeftBot, blk->LeftTop, blk->RightBot, blk->RightTop,
                             blk->TopLeft, blk->TopRight, blk->BotLeft, blk->BotRight};
        for (int k = 0; k < nblk; k++) {
            const int ib = blk->active[k];
            if (blk->level[ib] < c.minlevel || blk->level[ib] > c.maxlevel)
                return fail(BGF_ERR_INVALID_ARG, "block level outside the batch's range");
            for (auto* nb : nbs)
                if (nb[ib] < 0 || nb[ib] >= nbm || !seen[nb[ib]]) return fail(BGF_ERR_INVALID_ARG, "bad neighbour");
        }
    }
    for (int k = 0; !b->amr && k < nblk; k++) {
        const int ib = blk->active[k];
        if (blk->level[ib] != 0) return fail(BGF_ERR_UNSUPPORTED, "batch members must be one-level grids at level 0");
        const int* pairs[4][2] = {{blk->LeftBot, blk->LeftTop}, {blk->RightBot, blk->RightTop},
                                  {blk->TopLeft, blk->TopRight}, {blk->BotLeft, blk->BotRight}};
        for (auto& pr : pairs) {
            const int n0 = pr[0][ib], n1 = pr[1][ib];
            if (n0 < 0 || n0 >= nbm || !seen[n0] || n0 != n1 || blk->level[n0] != 0)
                return fail(BGF_ERR_UNSUPPORTED, "batch members must be one-level grids at level 0");
        }
    }
    int m = -1;
    for (int k = 0; k < b->cap_members; k++)
        if (!b->members[k].used) { m = k; break; }
    if (m < 0) return fail(BGF_ERR_OOM, "batch member capacity exhausted");
    int off = -1;  // first fit
    for (int k = 0, run = 0; k < b->cap_blocks; k++) {
        run = b->slot_owner[k] < 0 ? run + 1 : 0;
        if (run == nbm) { off = k - nbm + 1; break; }
    }
    if (off < 0) return fail(BGF_ERR_OOM, "batch block capacity exhausted");
    Member& M = b->members[m];
    M = Member();
    M.used = true;
    M.off = off;
    M.nblk = nblk;
    M.nblkmem = nbm;
    M.rain = (double)(float)p->rain;
    for (int k = 0; k < nblk; k++) M.active.push_back(off + blk->active[k]);
    if (b->amr) {
        M.order = M.active;  // the multi-level kernels keep the member's active order
        const int* nbs[8] = {blk->LeftBot, blk->LeftTop, blk->RightBot, blk->RightTop,
                             blk->TopLeft, blk->TopRight, blk->BotLeft, blk->BotRight};
        M.fix = fix_blocks(blk->active, nblk, blk->level, nbs, false, M.fix_all, M.odd);
        for (int& ib : M.fix) ib += off;
    } else {
        M.xy = block_xy(blk, nblk, p->dx);
        for (int& ib : M.xy.id) ib += off;
        M.order = processing_order(M.xy, b->tile_x, b->tile_y);
    }
    for (int k = 0; k < nbm; k++) b->slot_owner[off + k] = m;
    auto undo = [&](bgf_status e) {
        for (int k = 0; k < nbm; k++) b->slot_owner[off + k] = -1;
        b->members[m] = Member();
        return e;
    };
    // block description, offset into the range
    const int* nbs[8] = {blk->LeftBot, blk->LeftTop, blk->RightBot, blk->RightTop,
                         blk->TopLeft, blk->TopRight, blk->BotLeft, blk->BotRight};
    std::vector<int> tmp(nbm);
    for (int k = 0; k < 8; k++) {
        for (int i = 0; i < nbm; i++) tmp[i] = off + (seen[i] ? nbs[k][i] : i);
        if (hipMemcpy(b->d_nb[k] + off, tmp.data(), sizeof(int) * nbm, hipMemcpyHostToDevice) != hipSuccess)
            return undo(fail(BGF_ERR_HIP, "neighbour upload failed"));
    }
    for (int i = 0; i < nbm; i++) tmp[i] = b->amr && seen[i] ? blk->level[i] : 0;
    if (hipMemcpy(b->d_level + off, tmp.data(), sizeof(int) * nbm, hipMemcpyHostToDevice) != hipSuccess)
        return undo(fail(BGF_ERR_HIP, "level upload failed"));
    const size_t bytes = b->es * (size_t)nbm * BS, o = b->es * (size_t)off * BS;
    auto up = [&](void* dst, const void* src) {
        return hipMemcpy((char*)dst + o, src, bytes, hipMemcpyHostToDevice) == hipSuccess;
    };
    if (!(up(b->d_zb, zb) && up(b->d_h[0], hh) && up(b->d_u[0], u) && up(b->d_v[0], v) && up(b->d_cf, cf)))
        return undo(fail(BGF_ERR_HIP, "state upload failed"));
    if (hipMemset((char*)b->d_hmax + sizeof(float) * (size_t)off * BS, 0, sizeof(float) * (size_t)nbm * BS) !=
        hipSuccess)
        return undo(fail(BGF_ERR_HIP, "max-depth reset failed"));
    // the compensation array holds each block's interior only (BSI values per block)
    if (b->d_ch && hipMemset((char*)b->d_ch + b->es * (size_t)off * BSI, 0, b->es * (size_t)nbm * BSI) != hipSuccess)
        return undo(fail(BGF_ERR_HIP, "compensation reset failed"));
    s = rebuild(b);
    if (s != BGF_OK) return undo(s);
    const bgf::KParams P = member_view(b, m, active_offset(b, m));
    if (b->amr) {  // the bed's halo (InitzbHalo, src/InitialConditions.cu:135-147)
        bgf::launch_amr_fill(b->prec == 0 ? 0 : 1, P, b->d_zb, b->stream);
        HIPCHK(hipGetLastError());
    }
    // initial time step of the member (src/Mainloop.cu:515-554)
    bgf::DevLoop L = empty_loop();
    L.done = 0;
    L.nextoutputtime = endtime;
    L.endtime = endtime;
    bgf::set_rain(L, M.rain);
    L.dtmax = dtinit > 0 ? dtinit / 1.5 : level_dx(p->delta, b->amr ? p->maxlevel : 0) / std::sqrt(p->g * 10.0);
    HIPCHK(hipMemcpy(b->d_loop + m, &L, sizeof(L), hipMemcpyHostToDevice));
    bgf::launch_init_dt_member(b->prec, P, b->d_h[0], b->d_loop, m, b->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(&L, b->d_loop + m, sizeof(L), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    L.dtmax = L.dt;
    L.dt = 0.0;
    L.steps_done = 0;
    L.nstep = 0;
    L.gevery = 0;
    std::vector<int> nog(NGAUGE, -1);
    HIPCHK(hipMemcpy(b->d_gcell + NGAUGE * m, nog.data(), sizeof(int) * NGAUGE, hipMemcpyHostToDevice));
    L.done = L.totaltime >= L.endtime ? 1 : 0;
    // a roughness that is one value over the member's active cells reaches the corrector as that value
    L.cf_uniform = 1;
    for (int ibl = 0; L.cf_uniform && ibl < p->nblk; ibl++) {
        const int ib = blk->active[ibl];
        for (int j = 0; L.cf_uniform && j < BW; j++)
            for (int i = 0; i < BW; i++) {
                const size_t n = (size_t)memloc(i, j, ib);
                const double c = b->prec == 0 ? ((const double*)cf)[n] : (double)((const float*)cf)[n];
                if (ibl == 0 && i == 0 && j == 0) L.cf_value = c;
                else if (!(c == L.cf_value) || std::signbit(c) != std::signbit(L.cf_value)) { L.cf_uniform = 0; break; }
            }
    }
    if (!L.cf_uniform) L.cf_value = 0.0;
    b->loops[m] = L;
    *member = m;
    return BGF_OK;
}

bgf_status bgf_batch_remove(bgf_batch b, int m) {
    bgf_status s = check_member(b, m);
    if (s != BGF_OK) return s;
    Member& M = b->members[m];
    for (int k = 0; k < M.nblkmem; k++) b->slot_owner[M.off + k] = -1;
    M = Member();
    b->loops[m] = empty_loop();
    return rebuild(b);
}

bgf_status bgf_batch_run_async(bgf_batch b, int nsteps) {
    if (!b || nsteps < 0) return fail(BGF_ERR_INVALID_ARG, "bad argument");
    if (b->pending) return fail(BGF_ERR_STATE, "bgf_batch_run_async pending: call bgf_batch_sync first");
    for (auto& L : b->loops) {
        L.steps_done = 0;
        L.go = 0;
        for (int k = 0; k < bgf::NSLOT; k++) {
            L.slot32[k] = 0x7f800000u;
            L.slot64[k] = 0x7ff0000000000000ull;
        }
    }
    bgf_status s = prepare_run(b);
    if (s != BGF_OK) return s;
    HIPCHK(hipMemcpyAsync(b->d_loop, b->loops.data(), sizeof(bgf::DevLoop) * b->cap_members, hipMemcpyHostToDevice,
                          b->stream));
    if (b->krun.nblk > 0) {
        if (b->use_graph && nsteps >= 2 * PERIOD) {
            if (!b->graph) {
                hipGraph_t g = nullptr;
                HIPCHK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
                enqueue_steps(b, PERIOD);
                HIPCHK(hipStreamEndCapture(b->stream, &g));
                hipError_t e = hipGraphInstantiate(&b->graph, g, nullptr, nullptr, 0);
                (void)hipGraphDestroy(g);
                if (e != hipSuccess) {
                    b->graph = nullptr;
                    return fail(BGF_ERR_HIP, std::string("hipGraphInstantiate: ") + hipGetErrorString(e));
                }
            }
            for (int k = 0; k < nsteps / PERIOD; k++) HIPCHK(hipGraphLaunch(b->graph, b->stream));
            nsteps %= PERIOD;
        }
        enqueue_steps(b, nsteps);
    }
    HIPCHK(hipGetLastError());
    b->pending = 1;
    return BGF_OK;
}

bgf_status bgf_batch_sync(bgf_batch b) {
    if (!b) return fail(BGF_ERR_INVALID_ARG, "null batch");
    if (!b->pending) return fail(BGF_ERR_STATE, "nothing pending");
    b->pending = 0;
    HIPCHK(hipMemcpyAsync(b->loops.data(), b->d_loop, sizeof(bgf::DevLoop) * b->cap_members, hipMemcpyDeviceToHost,
                          b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    if (b->nactive_blocks > 0 && !b->amr) {  // multi-level members end every step in buffer 0
        const void* src[3] = {b->d_h[1], b->d_u[1], b->d_v[1]};
        void* dst[3] = {b->d_h[0], b->d_u[0], b->d_v[0]};
        bgf::launch_settle(b->prec, b->kp, src, dst, b->d_loop, nullptr, b->stream);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(b->stream));
    }
    int bad = 0;
    for (int m = 0; m < b->cap_members; m++) {
        if (!b->members[m].used) continue;
        b->cell_updates += (long long)b->loops[m].steps_done * b->members[m].nblk * BW * BW;
        bad |= b->loops[m].bad;
    }
    if (bad) return fail(BGF_ERR_NONFINITE_DT, "non-finite or non-positive time step in a member");
    return BGF_OK;
}

bgf_status bgf_batch_loop(bgf_batch b, int m, bgf_loop* loop, int* done) {
    bgf_status s = check_member(b, m);
    if (s != BGF_OK) return s;
    const bgf::DevLoop& L = b->loops[m];
    if (loop) {
        loop->nextoutputtime = L.nextoutputtime;
        loop->dt = L.dt;
        loop->dtmax = L.dtmax;
        loop->totaltime = L.totaltime;
    }
    if (done) *done = L.done;
    return BGF_OK;
}

bgf_status bgf_batch_get_state(bgf_batch b, int m, void* zs, void* hh, void* u, void* v) {
    bgf_status s = check_member(b, m);
    if (s != BGF_OK) return s;
    const Member& M = b->members[m];
    void* const dst[4] = {zs, hh, u, v};
    int most = 0;
    for (const Member& x : b->members)
        if (x.used) most = std::max(most, x.nblk);
    return read_back(*b->back, b->prec, M.active, most, M.off, b->d_active + active_offset(b, m), b->d_zb, b->d_h[0],
                     b->d_u[0], b->d_v[0], dst, b->stream);
}

bgf_status bgf_batch_volume(bgf_batch b, int m, double* volume) {
    bgf_status s = check_member(b, m);
    if (s != BGF_OK || !volume) return s != BGF_OK ? s : fail(BGF_ERR_INVALID_ARG, "null argument");
    const bgf::KParams P = member_view(b, m, active_offset(b, m));
    bgf::launch_volume(b->prec, P, b->d_h[0], b->d_volpart, b->d_volout, b->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(volume, b->d_volout, sizeof(double), hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return BGF_OK;
}

bgf_status bgf_batch_update_maxdepth(bgf_batch b) {
    if (!b) return fail(BGF_ERR_INVALID_ARG, "null batch");
    if (b->pending) return fail(BGF_ERR_STATE, "bgf_batch_run_async pending: call bgf_batch_sync first");
    if (b->nactive_blocks > 0) {
        bgf::launch_maxdepth(b->prec, b->kp, b->d_h[0], (float*)b->d_hmax, b->stream);
        HIPCHK(hipGetLastError());
    }
    return BGF_OK;
}

bgf_status bgf_batch_get_maxdepth(bgf_batch b, int m, float* hmax) {
    bgf_status s = check_member(b, m);
    if (s != BGF_OK || !hmax) return s != BGF_OK ? s : fail(BGF_ERR_INVALID_ARG, "null argument");
    const Member& M = b->members[m];
    HIPCHK(hipMemcpyAsync(hmax, (const float*)b->d_hmax + (size_t)M.off * BS, sizeof(float) * (size_t)M.nblkmem * BS,
                          hipMemcpyDeviceToHost, b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    return BGF_OK;
}

bgf_status bgf_batch_set_gauges(bgf_batch b, int m, int n, const int* cells, int every) {
    bgf_status s = check_member(b, m);
    if (s != BGF_OK) return s;
    Member& M = b->members[m];
    if (n < 0 || n > NGAUGE || (n > 0 && !cells)) return fail(BGF_ERR_INVALID_ARG, "at most 16 gauges");
    if (every < 0) return fail(BGF_ERR_INVALID_ARG, "bad sampling period");
    b->loops[m].gevery = n > 0 ? every : 0;
    if (n > 0 && every > 0 && !b->gauges_on) {
        b->gauges_on = true;
        b->run_valid = false;  // the captured step gains the sampling kernel
    }
    std::vector<int> g(NGAUGE, -1);
    M.gauges.clear();
    for (int k = 0; k < n; k++) {
        if (cells[k] < 0 || cells[k] >= M.nblkmem * BS) return fail(BGF_ERR_INVALID_ARG, "gauge cell out of range");
        g[k] = M.off * BS + cells[k];
        M.gauges.push_back(g[k]);
    }
    HIPCHK(hipMemcpy(b->d_gcell + NGAUGE * m, g.data(), sizeof(int) * NGAUGE, hipMemcpyHostToDevice));
    return BGF_OK;
}

bgf_status bgf_batch_sample_gauges(bgf_batch b, float* values, double* times) {
    if (!b || !values) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (b->pending) return fail(BGF_ERR_STATE, "bgf_batch_run_async pending: call bgf_batch_sync first");
    bgf::launch_gauges(b->prec, b->d_h[0], b->d_gcell, b->d_gval, NGAUGE * b->cap_members, b->stream);
    HIPCHK(hipGetLastError());
    HIPCHK(hipMemcpyAsync(values, b->d_gval, sizeof(float) * NGAUGE * b->cap_members, hipMemcpyDeviceToHost,
                          b->stream));
    HIPCHK(hipStreamSynchronize(b->stream));
    if (times)
        for (int m = 0; m < b->cap_members; m++) times[m] = b->loops[m].totaltime;
    return BGF_OK;
}

bgf_status bgf_batch_get_gauges(bgf_batch b, int m, float* values, double* times, int* nsamples) {
    bgf_status s = check_member(b, m);
    if (s != BGF_OK) return s;
    const bgf::DevLoop& L = b->loops[m];
    const int n = L.gevery > 0 ? std::min(NSAMP, L.nstep / L.gevery) : 0;
    if (nsamples) *nsamples = n;
    if (n > 0 && values)
        for (int g = 0; g < NGAUGE; g++)
            HIPCHK(hipMemcpy(values + (size_t)g * NSAMP, b->d_ring + ((size_t)m * NGAUGE + g) * NSAMP,
                             sizeof(float) * n, hipMemcpyDeviceToHost));
    if (n > 0 && times)
        HIPCHK(hipMemcpy(times, b->d_tring + (size_t)m * NSAMP, sizeof(double) * n, hipMemcpyDeviceToHost));
    return BGF_OK;
}

bgf_status bgf_batch_track_maxdepth(bgf_batch b, int on) {
    if (!b) return fail(BGF_ERR_INVALID_ARG, "null batch");
    if (b->pending) return fail(BGF_ERR_STATE, "bgf_batch_run_async pending: call bgf_batch_sync first");
    b->track_max = on != 0;
    b->run_valid = false;
    return BGF_OK;
}

bgf_status bgf_batch_stats(bgf_batch b, long long* cell_updates, int* nmembers, int* nblocks) {
    if (!b) return fail(BGF_ERR_INVALID_ARG, "null batch");
    int n = 0;
    for (auto& M : b->members) n += M.used ? 1 : 0;
    if (cell_updates) *cell_updates = b->cell_updates;
    if (nmembers) *nmembers = n;
    if (nblocks) *nblocks = b->nactive_blocks;
    return BGF_OK;
}

bgf_status bgf_batch_set_schedule(bgf_batch b, int tile_x, int tile_y, int wg_pred, int wg_corr) {
    if (!b) return fail(BGF_ERR_INVALID_ARG, "null batch");
    if (b->pending) return fail(BGF_ERR_STATE, "bgf_batch_run_async pending: call bgf_batch_sync first");
    if (tile_x < 0 || tile_y < 0 || tile_x > 4096 || tile_y > 4096 || wg_pred < 0 || wg_corr < 0 || wg_pred > 64 ||
        wg_corr > 64)
        return fail(BGF_ERR_INVALID_ARG, "schedule out of range");
    const int tx = tile_x ? tile_x : b->tile_x, ty = tile_y ? tile_y : b->tile_y;
    if (tx != b->tile_x || ty != b->tile_y) {
        for (auto& M : b->members)
            if (M.used) M.order = processing_order(M.xy, tx, ty);
        b->tile_x = tx;
        b->tile_y = ty;
    }
    b->wg_pred = wg_pred;
    b->wg_corr = wg_corr;
    HIPCHK(hipStreamSynchronize(b->stream));
    return rebuild(b);  // re-uploads the order; the run set, grids and graph are redone on the next run
}

bgf_status bgf_batch_get_schedule(bgf_batch b, int* tile_x, int* tile_y, int* wg_pred, int* wg_corr) {
    if (!b) return fail(BGF_ERR_INVALID_ARG, "null batch");
    if (tile_x) *tile_x = b->tile_x;
    if (tile_y) *tile_y = b->tile_y;
    if (wg_pred) *wg_pred = b->wg_pred;
    if (wg_corr) *wg_corr = b->wg_corr;
    return BGF_OK;
}

}  // extern "C"
