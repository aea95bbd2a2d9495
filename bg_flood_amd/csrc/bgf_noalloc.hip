// bgf_noalloc.hip -- the one-level step for callers that cannot allocate
// device memory (bgf_step_noalloc).
//
// The step's own scratch -- the predictor's tendencies dh, dhu, dhv, the
// block records of the persistent kernels, their work-queue counters and the
// device loop state with its dt slots -- lives in one file-scope device array
// (`scratch`, SCRATCH_BYTES per GPU, held by every GPU the library runs on
// until the process ends).  Host code never passes the array's name to a
// kernel or a copy: the name is a host-side stand-in, not a device address.
// Its address on each device is taken once, with hipGetSymbolAddress, at the
// entry point's first call on that device, and that address is what the
// kernels receive.  Everything else -- the state, the bed, the roughness, the
// block description and the result -- is the caller's device memory.
//
// Every call on a GPU shares that GPU's array and finds the contents the last
// call left: the queue counters, which must start at zero, are cleared when
// the address is taken and are left at zero by every step (each persistent
// kernel zeroes the other's counters), and the loop state is written at the
// start of each call.  Calls that overlap on one GPU (two host threads, or two
// streams in flight) race on the array.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "bgf_host.h"
#include "bgf_kernels.h"

using namespace bgf_host;

namespace {

constexpr size_t SCRATCH_BYTES = size_t(64) << 20;  // 64 MiB per GPU
constexpr int MAX_DEVICES = 64;

static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

// Byte offsets of the scratch regions for nblk blocks in `slots` block slots
// and values of es bytes, each region 256-byte aligned.  The block records go
// by position in the block list, the tendencies by block slot: the kernels
// address every cell array with the slot, and a list may leave slots unused.
struct Layout {
    size_t loop, queue, rec, dh, dhu, dhv, end;
};
inline size_t up256(size_t n) { return (n + 255) / 256 * 256; }
Layout layout(long long nblk, long long slots, size_t es) {
    Layout L;
    L.loop = 0;
    L.queue = up256(2 * sizeof(bgf::DevLoop));  // the step's loop state and the one that it leaves
    L.rec = L.queue + up256(sizeof(int) * 2 * bgf::NXCD * bgf::QSTRIDE);
    const size_t tend = up256((size_t)slots * BSI * es);
    L.dh = L.rec + up256((size_t)nblk * 8 * sizeof(int));
    L.dhu = L.dh + tend;
    L.dhv = L.dhu + tend;
    L.end = L.dhv + tend;
    return L;
}
// The largest count of blocks, without unused slots, whose regions fit the array.
long long max_blocks(size_t es) {
    long long lo = 0, hi = (long long)(SCRATCH_BYTES / (BSI * es)) + 1;
    while (hi - lo > 1) {
        const long long mid = (lo + hi) / 2;
        (layout(mid, mid, es).end <= SCRATCH_BYTES ? lo : hi) = mid;
    }
    return lo;
}

// Clears n ints (the queue counters): a kernel rather than a memset, so the
// clearing is an ordinary launch wherever the call happens.
__global__ void k_zero_ints(int* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// The loop state of one step (what bgf_step uploads): the caller's Loop<T>,
// the uniform rain rate, every dt slot empty.
__global__ void k_loop_state(bgf::DevLoop* L, double nextoutputtime, double dt, double dtmax, double totaltime,
                             double rain_mmh, float rate32, double dtmin) {
    const int t = threadIdx.x;
    if (t == 0) {
        L->nextoutputtime = nextoutputtime;
        L->dt = dt;
        L->dtmax = dtmax;
        L->totaltime = totaltime;
        L->endtime = 1e300;
        L->rain = rain_mmh;
        L->rate64 = rain_mmh / 1000.0 / 3600.0;
        L->rate32 = rate32;
        L->done = 0;
        L->bad = 0;
        L->steps_done = 0;
        L->go = 0;
        L->nstep = 0;
        L->gevery = 0;
        L->rain_t = nullptr;
        L->rain_v = nullptr;
        L->rain_n = 0;
        L->tcorr = 0.0;
        L->tpred = 0.0;
        L->tstart = 0.0;
        L->stats_n = 0;
        L->cf_uniform = 0;
        L->cf_value = 0.0;
        L->dtmin = dtmin;
        L->crashed = 0;
        L->unused = 0;
    }
    if (t < bgf::NSLOT) {
        L->slot32[t] = 0x7f800000u;
        L->slot64[t] = 0x7ff0000000000000ull;
    }
}

std::mutex g_mu;
unsigned char* g_scratch[MAX_DEVICES] = {};

// The scratch array's address on the current device, taken (and its queue
// counters cleared) at the first call on that device.
bgf_status scratch_on_device(int dev, hipStream_t st, unsigned char** out) {
    if (dev < 0 || dev >= MAX_DEVICES) return fail(BGF_ERR_UNSUPPORTED, "device index above 63");
    std::lock_guard<std::mutex> lk(g_mu);
    if (!g_scratch[dev]) {
        unsigned char* ptr = nullptr;
        const hipError_t e = hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(BGF_ERR_HIP, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
        const Layout L = layout(0, 0, 4);
        const int nq = 2 * bgf::NXCD * bgf::QSTRIDE;
        hipLaunchKernelGGL(k_zero_ints, dim3((nq + 255) / 256), dim3(256), 0, st, (int*)(ptr + L.queue), nq);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(st));
        g_scratch[dev] = ptr;
    }
    *out = g_scratch[dev];
    return BGF_OK;
}

}  // namespace

extern "C" bgf_status bgf_step_noalloc(const bgf_param* p, const bgf_blocks* d_blocks, const void* zb, const void* cf,
                                       const void* hh, const void* u, const void* v, void* ho, void* uo, void* vo,
                                       bgf_loop* loop, void* stream) {
    bgf_status s = check_param(p);
    if (s != BGF_OK) return s;
    if (!d_blocks || !loop) return fail(BGF_ERR_INVALID_ARG, "null argument");
    if (p->precision == BGF_FP32_COMP)
        return fail(BGF_ERR_UNSUPPORTED, "BGF_FP32_COMP keeps a compensation per cell across steps: use a handle");
    if (p->spherical) return fail(BGF_ERR_UNSUPPORTED, "spherical grids need a handle (metric terms)");
    if (p->minlevel != p->maxlevel)
        return fail(BGF_ERR_UNSUPPORTED, "one-level meshes only (minlevel == maxlevel)");
    const size_t es = p->precision == BGF_FP64 ? 8 : 4;
    const long long maxb = max_blocks(es);
    if (p->nblk > maxb)
        return fail(BGF_ERR_INVALID_ARG, "nblk " + std::to_string(p->nblk) + " exceeds the " +
                                             std::to_string(maxb) + " blocks that the 64 MiB scratch array holds at "
                                             "this precision");
    const void* dev_ptrs[] = {d_blocks->active, d_blocks->LeftBot, d_blocks->RightBot, d_blocks->BotLeft,
                              d_blocks->TopLeft, zb, cf, hh, u, v, ho, uo, vo};
    for (const void* q : dev_ptrs)
        if (!device_accessible(q)) return fail(BGF_ERR_INVALID_ARG, "an array is not device memory");
    if (ho == hh || uo == u || vo == v) return fail(BGF_ERR_INVALID_ARG, "the result must not overwrite the input");
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    hipStream_t st = (hipStream_t)stream;
    unsigned char* base = nullptr;
    s = scratch_on_device(dev, st, &base);
    if (s != BGF_OK) return s;
    long long slots = p->nblkmem;
    if (layout(p->nblk, slots, es).end > SCRATCH_BYTES) {
        // the list may still use low slots only: those up to the greatest in it are needed
        std::vector<int> act(p->nblk);
        HIPCHK(hipMemcpyAsync(act.data(), d_blocks->active, sizeof(int) * act.size(), hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
        slots = *std::max_element(act.begin(), act.end()) + 1LL;
        if (layout(p->nblk, slots, es).end > SCRATCH_BYTES)
            return fail(BGF_ERR_INVALID_ARG, "a block in slot " + std::to_string(slots - 1) + ": the 64 MiB scratch "
                                             "array does not hold " + std::to_string(slots) +
                                             " block slots at this precision");
    }
    const Layout Lo = layout(p->nblk, slots, es);
    bgf::DevLoop* dL = (bgf::DevLoop*)(base + Lo.loop);

    bgf::KParams kp;
    std::memset(&kp, 0, sizeof(kp));
    kp.g = p->g; kp.eps = p->eps; kp.CFL = p->CFL; kp.theta = p->theta;
    kp.delta0 = p->delta;
    kp.delta = level_dx(p->delta, p->minlevel);
    kp.fc = p->precision == BGF_FP64 ? coriolis<double>(p->lat) : coriolis<float>(p->lat);
    kp.mask = p->mask;
    kp.rain_mmh = (double)(float)p->rain;  // Rain.nowvalue is a float (src/Forcing.h)
    kp.frictionmodel = p->frictionmodel;
    kp.aoibnd = p->aoibnd;
    kp.ForceMassConserve = p->ForceMassConserve;
    kp.rain_on = p->rain_on;
    kp.nblk = p->nblk;
    kp.wetdryfix = p->wetdryfix;
    kp.minlevel = kp.maxlevel = p->minlevel;
    kp.grid_pred = bgf::persistent_grid(p->precision, 0, p->nblk, 0);
    kp.grid_corr = bgf::persistent_grid(p->precision, 1, p->nblk, 0);
    if (kp.grid_pred <= 0 || kp.grid_corr <= 0) return fail(BGF_ERR_HIP, "occupancy query failed");
    kp.active = d_blocks->active;
    kp.order = d_blocks->active;  // processed in the active order
    kp.rec = (const int*)(base + Lo.rec);
    kp.queue = (int*)(base + Lo.queue);
    kp.LeftBot = d_blocks->LeftBot;
    kp.RightBot = d_blocks->RightBot;
    kp.BotLeft = d_blocks->BotLeft;
    kp.TopLeft = d_blocks->TopLeft;
    kp.level = d_blocks->level;

    bgf::launch_records(kp, (int*)(base + Lo.rec), st);
    const float r32 = (float)((float)p->rain / 1000.0f / 3600.0f);
    hipLaunchKernelGGL(k_loop_state, dim3(1), dim3(64), 0, st, dL, loop->nextoutputtime, loop->dt, loop->dtmax,
                       loop->totaltime, kp.rain_mmh, r32, p->dtmin);
    HIPCHK(hipGetLastError());
    alignas(16) unsigned char storage[sizeof(bgf::StepBuffers<double>)];
    if (p->precision == BGF_FP64) {
        auto* B = (bgf::StepBuffers<double>*)storage;
        B->h = (const double*)hh; B->u = (const double*)u; B->v = (const double*)v;
        B->ho = (double*)ho; B->uo = (double*)uo; B->vo = (double*)vo;
        B->zb = (const double*)zb; B->cf = (const double*)cf;
        B->dh = (double*)(base + Lo.dh); B->dhu = (double*)(base + Lo.dhu); B->dhv = (double*)(base + Lo.dhv);
        B->ch = nullptr;
    } else {
        auto* B = (bgf::StepBuffers<float>*)storage;
        B->h = (const float*)hh; B->u = (const float*)u; B->v = (const float*)v;
        B->ho = (float*)ho; B->uo = (float*)uo; B->vo = (float*)vo;
        B->zb = (const float*)zb; B->cf = (const float*)cf;
        B->dh = (float*)(base + Lo.dh); B->dhu = (float*)(base + Lo.dhu); B->dhv = (float*)(base + Lo.dhv);
        B->ch = nullptr;
    }
    bgf::launch_step(p->precision, kp, storage, dL, dL + 1, 0, st, nullptr);
    HIPCHK(hipGetLastError());
    bgf::DevLoop D;
    HIPCHK(hipMemcpyAsync(&D, dL + 1, sizeof(D), hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    loop->dt = D.dt;
    loop->dtmax = D.dtmax;
    if (D.bad) return fail(BGF_ERR_NONFINITE_DT, "non-finite or non-positive time step");
    return BGF_OK;
}
