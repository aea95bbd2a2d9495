// bgf_kernels.h -- types shared by the HIP kernels and the host library.
#pragma once
#include <hip/hip_runtime.h>

namespace bgf {

constexpr int NSLOT = 64;  // block-minimum dt slots (atomic min, spread to avoid contention)

// Device-resident Loop<T> time keeping (src/Arrays.h:358-366) and run flags.
struct LoopState {
    double nextoutputtime;
    double dt;
    double dtmax;
    double totaltime;
    double endtime;  // the run stops once totaltime reaches it
    double rain;     // uniform rain rate, mm/h (Rain.nowvalue)
    double rate64;   // T(rain) / T(1000) / T(3600) in FP64, and rate32 in FP32: the depth rate in m/s
                     // (src/Updateforcing.cu:559), formed once per loop instead of per cell
    double tcorr;    // time of the corrector's boundary values: the step's start + dt (set by the dt reduction)
    double tpred;    // time of the predictor's boundary fluxes: the step's start + half the previous dt (set
                     // by the dt reduction before it replaces dt; multi-level kernels read it after it)
    double tstart;   // time at the step's start (set by the dt reduction)
    double cf_value; // batch member: the roughness where cf_uniform is set
    double dtmin;    // Param.dtmin: a run stops after a step with dt < dtmin before its end time (0: never)
    // uniform rain as a time series (rain_n > 0): the rate of each step is
    // interpolated at its start by the dt reduction, which sets rate64/rate32
    const double* rain_t;
    const double* rain_v;
    int rain_n;
    float rate32;
    int done;        // totaltime reached the end time: later steps are no-ops
    int bad;         // a non-finite or non-positive dt was produced
    int steps_done;  // steps executed since the loop was uploaded
    int go;          // set by the dt reduction: the corrector half of this step runs
    int nstep;       // steps since the domain started (gauge sampling counts these)
    int gevery;      // gauge sampling period in steps (batch members)
    int stats_n;     // steps since the output statistics' means were reset (Loop.nstep of Calcmeanmax)
    int cf_uniform;  // batch member: every active cell has roughness cf_value (the corrector skips the cf array)
    int crashed;     // the run stopped on dtmin (CrashDetection, src/Mainloop.cu:648-660)
    int unused;      // keeps the size a multiple of eight, so copies leave no padding behind
};
// A loop state with the dt reduction's slots (bit patterns of positive floats; +inf when empty).
// A single domain has two: a step's predictor fills the slots of the first, its later launches
// each work the new state out from them, and one workgroup leaves it, with empty slots, in the
// second, which the next step takes as its first.  A batch has one per member, reduced in place.
struct DevLoop : LoopState {
    unsigned int slot32[NSLOT];
    unsigned long long slot64[NSLOT];
};

// Sets a loop state's rain rate and its per-second depth rates.
inline void set_rain(LoopState& L, double rain_mmh) {
    L.rain = rain_mmh;
    L.rate64 = rain_mmh / 1000.0 / 3600.0;
    volatile float r = (float)rain_mmh;  // each division rounded to float, as on the device
    r = r / 1000.0f;
    r = r / 3600.0f;
    L.rate32 = r;
}

// Scalar parameters and block neighbour arrays of one domain.
// A boundary segment on the device (bndsegment, src/Forcing.h:130-150): its
// type; its water level from a uniform series (n pairs of time t, level z),
// from a level map (now: the map at the step's start, nx*ny levels, x fastest,
// on the grid from (xo, yo) by (dx, dy); frames: nt maps at to + k*tdt that it
// is interpolated from, or null when the caller keeps now current), or zs0 (a
// segment without forcing, Param.zsinit or 0); on: it has forcing, and ramps
// in with the taper.
struct BSeg {
    const double* t;
    const double* z;
    const float* frames;
    float* now;
    double xo, yo, dx, dy, to, tdt, zs0;
    int type, n, nx, ny, nt, on;
};

struct KParams {
    double g, eps, CFL, theta;
    double delta;   // cell size of the one-level kernels' level
    double delta0;  // Param.delta: cell size of level 0
    double fc, mask, rain_mmh;
    int frictionmodel, aoibnd, ForceMassConserve, rain_on, nblk, wetdryfix;
    int grid_pred, grid_corr;  // persistent workgroup counts (multiples of 8)
    int* queue;                // the persistent kernels' 16 work-queue counters, QSTRIDE apart (zeroed at allocation)
    int cf_uniform;            // every active cell has roughness cf_value: the one-level corrector skips the cf array
    double cf_value;
    const int* active;  // active blocks in the reference order
    const int* order;   // the same blocks in the persistent kernels' processing order
    const int* rec;     // per position of the order: block, LeftBot, RightBot, BotLeft, TopLeft, member, 0, 0
    const int* LeftBot;
    const int* RightBot;
    const int* BotLeft;
    const int* TopLeft;
    // multi-level meshes
    const int* level;     // block level (every mesh)
    const int* LeftTop;
    const int* RightTop;
    const int* TopRight;
    const int* BotRight;
    const int* inv;       // position of each block in the active list (-1 if inactive)
    const int* nbr;       // per block slot, NBR ints (multi-level meshes; launch_amr_nbr): the eight
                          // neighbours LeftBot, LeftTop, RightBot, RightTop, BotLeft, BotRight,
                          // TopLeft, TopRight, then for each of them its level (low 8 bits, signed)
                          // and, in bit 8, whether the block is the first-half neighbour of the
                          // neighbour's side facing it, and of the block itself, in every one of
                          // them, whether it has a finer neighbour and a side on the domain edge
    // multi-level meshes: the active blocks whose advance waits for other blocks' faces
    // (nfix of them; fix_all: every block does)
    const int* fix;
    const int4* rcell;    // RECIPES per block slot: the cells a stage gathers (multi-level meshes; launch_amr_nbr)
    const int2* rmeta;    // and how it combines them
    int odd;              // a side's first neighbour is not finer than the block and its second is: no quadtree
    int nfix, fix_all;
    int minlevel, maxlevel;  // levels present among the active blocks
    // batches of domains: member of each block (DevLoop of that member), member count
    const int* sid;
    int nmember;
    // spherical grids: per-block rows of metric terms in T (METRIC_STRIDE per block)
    const void* metric;
    int spherical;
    // running maximum depth of the interior cells, updated by every corrector (optional)
    float* hmax;
    // rain on a grid (optional): frames of rates [mm/h] (nx*ny each) at t0 + k*dtf,
    // the map of the current step (written at its start), and what the cells
    // need to sample it: Param.xo/yo/dx and the block origins
    const float* rframes;
    float* rnow;
    int rnx, rny, rnframes;
    double rxo, ryo, rdx, rt0, rdtf;
    double xo, yo, dx;
    const double* bxo;
    const double* byo;
    // boundary segments (optional): bseg[ib] is the segment of boundary block
    // ib, whose type and level all its boundary faces take; seg[] holds the
    // segments, the remainder (type aoibnd) last, nseg of them; without them
    // every boundary face is of type aoibnd.  Types: 0 wall, 1 Neumann (and 4),
    // 2 Dirichlet water level, 3 absorbing.  bmapmax: the largest level map.
    const unsigned char* bseg;
    const BSeg* seg;
    int nseg, bmapmax;
    int bopen;  // some segment has type 2 or 3
    // Param.zsoffset (added to the boundary level, as a float), Param.bndtaper and Param.inittime
    // (the level ramps from the inside water level over bndtaper seconds from inittime; 0: none)
    double bzsoffset, btaper, binittime;
    // river discharges (nriver > 0): each river's box (xstart, xend, ystart,
    // yend), flow series (time rt, flow rq from roff[r] to roff[r+1]), its
    // discharge area, and the blocks that may receive water
    int nriver;
    const double* rbox;
    const double* rt;
    const double* rq;
    const int* roff;
    const double* rarea;
    const unsigned char* rblk;
};

// Layout of a block's metric terms (spherical grids, src/Spherical.cu:15-64):
// cm of the X faces by row, cm and fm of the Y faces by face row (17), and for
// the tendencies cm, fm of the faces below and above, and the Coriolis factor.
enum { MET_CMX = 0, MET_CMY = 16, MET_FMY = 33, MET_CME = 50, MET_FMV = 66, MET_FMVP = 82, MET_FC = 98,
       METRIC_STRIDE = 128 };

constexpr int NXCD = 8;     // XCDs of an MI355X, each with its own L2
constexpr int QSTRIDE = 64; // ints between work-queue counters (a 256-byte line each)

template <class T> struct StepBuffers {
    const T* h;
    const T* u;
    const T* v;
    T* ho;
    T* uo;
    T* vo;
    const T* zb;
    const T* cf;
    T* dh;
    T* dhu;
    T* dhv;
    T* ch;  // compensation of h (BGF_FP32_COMP): the low-order part lost by the last updates
};

// ev (optional): four events recorded before the predictor, after it, after
// the reduction and after the corrector.  L: the step's loop state, Lnext: the
// next step's.  With P.sid set, the block list packs P.nmember domains, L holds
// one loop state per member, and Lnext is not used.
void launch_step(int precision, const KParams& P, const void* buffers, DevLoop* L, DevLoop* Lnext,
                 int advance_time, hipStream_t st, hipEvent_t* ev);
// Workgroups of a persistent launch; wg_per_cu > 0 caps the resident workgroups per CU.
int persistent_grid(int precision, int corrector, int nblk, int wg_per_cu);
void launch_init_dt(int precision, const KParams& P, const void* h, DevLoop* L, hipStream_t st);
// Fills rec (8 ints per position, 32-byte aligned) from P.order, the neighbour arrays and P.sid;
// called whenever the order, the mesh or the membership changes.
void launch_records(const KParams& P, int* rec, hipStream_t st);
// Initial dt of one member of a batch: P restricted to the member's blocks.
void launch_init_dt_member(int precision, const KParams& P, const void* h, DevLoop* L, int member, hipStream_t st);
// hmax = max(hmax, h) over the interior cells of P's blocks.
void launch_maxdepth(int precision, const KParams& P, const void* h, float* hmax, hipStream_t st);
// val[k] = h[cell[k]] (NaN where cell[k] < 0), k < n.
void launch_gauges(int precision, const void* h, const int* cell, float* val, int n, hipStream_t st);
// After a batch step: members that stepped record h at their 16 gauges every L.gevery of their own
// steps into ring[(m*16+g)*cap + k] and the time into tring[m*cap + k].
void launch_gauge_step(int precision, const void* h, const int* cell, const DevLoop* L, int nmember, int cap,
                       float* ring, double* tring, hipStream_t st);
void launch_volume(int precision, const KParams& P, const void* h, double* part, double* out, hipStream_t st);
// Copies h, u, v from src to dst for the blocks whose member ran an odd number of steps.
void launch_settle(int precision, const KParams& P, const void* const* src, void* const* dst, const DevLoop* L,
                   LoopState* out, hipStream_t st);
// The loop state S to L, with empty slots; and L's state to out, host memory the GPU can write, which
// launch_settle and launch_export do as well where out is not null.
void launch_set_loop(const LoopState& S, DevLoop* L, hipStream_t st);
void launch_loop_out(const DevLoop* L, LoopState* out, hipStream_t st);

// Interior cells of the active blocks: dst[0..2] = src[0..2] (h, u, v).
void launch_import(int precision, const KParams& P, const void* const* src, void* const* dst, hipStream_t st);
// Interior cells: dst = (h, zb + h, u, v) of src = (h, u, v); keep (may be null) receives h, u, v too.
void launch_export(int precision, const KParams& P, const void* const* src, const void* zb, void* const* dst,
                   void* const* keep, const DevLoop* L, LoopState* lout, hipStream_t st);

// Interior cells of the n blocks active[0..n) to out (host memory the GPU can write): block by block
// the fields whose bit is set in fields (0 zs = zb + h, 1 h, 2 u, 3 v), 256 values each.
void launch_pack_state(int precision, const int* active, int n, const void* zb, const void* h, const void* u,
                       const void* v, int fields, void* out, hipStream_t st);

// Refinement criteria (src/AdaptCriteria.cu:62-160) per active block of P:
// flags[ib] = any interior cell of a (plus b when b is not null: zs = zb + h)
// exceeds lo (mode 0) or lies in [lo, hi] (mode 1).
void launch_refine_flags(int precision, const KParams& P, const void* a, const void* b, int mode, double lo,
                         double hi, unsigned char* flags, hipStream_t st);

// dt reduction of the block-minimum slots, clamp and output landing (one wave per loop state), from
// L to Lnext (which may be L).
void launch_reduce_dt(int precision, DevLoop* L, DevLoop* Lnext, int nloop, int advance_time, hipStream_t st);

// Arrays of the multi-level step (the reference's Model<T> layout).
template <class T> struct AmrBuffers {
    T *h, *u, *v;     // evolv
    T *ho, *uo, *vo;  // evolv_o
    T* zb;            // its halo is written by the halo fill and the wet/dry prolongation
    const T* cf;
    T *Fhu, *Fqux, *Su, *Fqvx, *Fhv, *Fqvy, *Sv, *Fquy;  // face fluxes (no slope is stored)
    T* hsnap;         // h before the wet/dry prolongation (meshes of four levels and more)
    T *dh, *dhu, *dhv; // tendencies, interior cells only
};
// One step on a multi-level mesh: precision 0 FP64 and 1 FP32 in the reference
// arithmetic; 2 and 3 (BGF_FP32_FAST, BGF_FP32_COMP) FP32 with hardware
// reciprocals and square roots in the slopes and the fluxes.
void launch_amr_step(int precision, const KParams& P, const void* buffers, DevLoop* L, DevLoop* Lnext,
                     int advance_time, hipStream_t st, hipEvent_t* ev);
// Fills nbr (NBR ints per block slot, nbm slots) from P's eight neighbour arrays
// and the levels; slots whose neighbours are outside [0, nbm) get level 0.
constexpr int NBR = 16;
// Flags beside the level (low 8 bits) in a record's level words.
enum { REC_BACK = 1 << 8, REC_FINER = 1 << 9, REC_EDGE = 1 << 10 };
// and then the gather recipes of P's active blocks (RECIPES entries of cells and codes per block slot).
constexpr int RECIPES = 132;
void launch_amr_nbr(const KParams& P, int* nbr, int nbm, int4* rcell, int2* rmeta, hipStream_t st);
// Halo of a static field (the bed) on a multi-level mesh, src/InitialConditions.cu:135-147.
void launch_amr_fill(int precision, const KParams& P, void* z, hipStream_t st);
// The rain map of the coming step from the rain frames, and the boundary level
// maps of the coming step (nothing without frames).
void launch_rain_now(const KParams& P, const DevLoop* L, hipStream_t st);
// The step's halo fill of h, u, v on a multi-level mesh (src/Halo.cu:586-616) by itself.
void launch_amr_halo(int precision, const KParams& P, void* h, void* u, void* v, const void* zb, hipStream_t st);

// State of a multi-level mesh moved onto an adapted mesh (bgf_remesh.hip).
struct RemeshLaunch {
    int nblk;                             // active blocks of the new mesh
    const void *h, *u, *v, *zb, *cf;      // old state
    const int* active;                    // new mesh
    const int* level;
    const double *xo, *yo;
    const int* remap;                     // kind, src0..src3 per new slot
    void *nh, *nu, *nv, *nzb, *ncf;       // new state
    const float* bed;                     // bed source raster (may be null)
    int bnx, bny;
    double bxo, byo, bdx, pxo, pyo, dx, eps;
};
void launch_remesh(int precision, const KParams& Po, const RemeshLaunch& R, hipStream_t st);

// Output statistics of Calcmeanmax (src/Meanmax.cu:15-112) over the active blocks after a step.
struct StatsLaunch {
    int mask;              // 1 means, 2 maxima, 4 wet time
    double wet_threshold;  // Param.wet_threshold
    void* a[15];           // mean h, zs, u, v, U, hU, hUU; max h, zs, u, v, U, hU, hUU; wet time
};
// advanced: the step advanced totaltime (else the statistics take totaltime + dt as the step's end).
void launch_stats(int precision, const KParams& P, const StatsLaunch& S, const void* h, const void* u, const void* v,
                  const void* zb, const DevLoop* L, int advanced, hipStream_t st);
// Resets the statistics selected by `which` (1 means to 0, 2 maxima to -max(T), 4 wet time to 0).
void launch_stats_reset(int precision, const KParams& P, const StatsLaunch& S, int which, hipStream_t st);
// R.bed sampled onto the interior cells of R's mesh (R.active, level, xo, yo): R.nzb = interp2BUQ
// of the raster at every cell (only the raster, mesh and output fields of R are read).
void launch_sample_raster(int precision, const RemeshLaunch& R, hipStream_t st);

}  // namespace bgf
