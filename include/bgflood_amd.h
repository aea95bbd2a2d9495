/*
 * bgflood_amd.h -- C ABI of the MI355X-native BG_Flood timestep library.
 *
 * The library replaces the per-timestep shallow-water update of BG_Flood,
 * FlowGPU<T> / FlowCPU<T> (src/FlowGPU.cu:14-315, src/FlowCPU.cu:15-253), on
 * its block-uniform quadtree: 16x16-cell blocks stored with a one-cell halo
 * in 18x18 tiles, index (i+1) + (j+1)*18 + ib*324 (src/MemManagement.cu:37-40).
 * All arguments are plain pointers and sizes; no C++ or torch types cross it.
 * Every entry point returns a bgf_status; none calls exit().
 */
#ifndef BGFLOOD_AMD_H
#define BGFLOOD_AMD_H

#include <stddef.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Error codes.  The reference has none: CUDA_CHECK prints and exits
 * (src/Setup_GPU.cu:169-182). */
typedef enum {
    BGF_OK = 0,
    BGF_ERR_INVALID_ARG = 1,
    BGF_ERR_OOM = 2,
    BGF_ERR_HIP = 3,
    BGF_ERR_NONFINITE_DT = 4,
    BGF_ERR_UNSUPPORTED = 5,
    BGF_ERR_NO_DEVICE = 6,
    BGF_ERR_STATE = 7,
    BGF_ERR_CRASHED = 8   /* a step's dt fell below Param.dtmin before the end time: the run
                             stopped there, as CrashDetection stops the model
                             (src/Mainloop.cu:648-660) */
} bgf_status;

/* Arithmetic of a handle.  The reference picks T from Param.doubleprecision
 * (src/BG_Flood.cu:101-109). */
typedef enum {
    BGF_FP64 = 0,       /* T = double, operation-for-operation the reference CPU step */
    BGF_FP32 = 1,       /* T = float,  operation-for-operation the reference CPU step */
    BGF_FP32_FAST = 2,  /* T = float, hardware reciprocal / square root, fused multiply-add
                           (multi-level meshes: hardware reciprocal / square root in the
                           slopes and fluxes, the rest as BGF_FP32) */
    BGF_FP32_COMP = 3   /* BGF_FP32_FAST with the depth update accumulated in a compensated
                           (Kahan) sum: one more float per cell.  Multi-level meshes run
                           the multi-level BGF_FP32_FAST arithmetic for it. */
} bgf_precision;

/* Subset of class Param (src/Param.h:10-239) that the Kurganov step reads. */
typedef struct {
    double g;             /* Param.g */
    double eps;           /* Param.eps, drying height */
    double CFL;           /* Param.CFL */
    double theta;         /* Param.theta, minmod2 limiter parameter */
    double dx;            /* Param.dx */
    double delta;         /* Param.delta (== dx on Cartesian grids) */
    double xo, yo;        /* Param.xo, Param.yo */
    double lat;           /* Param.lat (Coriolis on Cartesian grids) */
    double mask;          /* Param.mask: cells with zb >= mask get no rain */
    int frictionmodel;    /* Param.frictionmodel: -1 Manning, 0 quadratic, 1 Smart */
    int engine;           /* Param.engine: only 2 (Kurganov) is provided */
    int aoibnd;           /* Param.aoibnd: remainder boundary type, 0 wall, 1 Neumann */
    int ForceMassConserve;/* Param.ForceMassConserve */
    int wetdryfix;        /* Param.wetdryfix */
    int spherical;        /* Param.spherical: lat/lon grid, dx in degrees, delta = dx*Radius*pi/180 */
    int nblk;             /* Param.nblk: active blocks */
    int nblkmem;          /* Param.nblkmem: allocated blocks (>= nblk) */
    int minlevel, maxlevel;
    int rain_on;          /* a uniform rain forcing is present (Forcing.Rain) */
    double rain;          /* Rain.nowvalue, mm/h */
    int precision;        /* bgf_precision */
    double Radius;        /* Param.Radius: sphere radius for spherical grids (6371220 m) */
    double dtmin;         /* Param.dtmin (src/Param.h:85, 0.0005 s in the reference): bgf_run
                             stops with BGF_ERR_CRASHED after a step whose dt is below it while
                             totaltime < endtime; <= 0 turns the check off */
} bgf_param;

/* BlockP<T> (src/Arrays.h:233-249): nblkmem entries each; active[ibl] for
 * ibl < nblk gives the block index ib.  A neighbour equal to the block itself
 * means "no neighbour" (src/Mesh.cu:390-397).  xo/yo are block origins. */
typedef struct {
    const int* active;
    const int* level;
    const int *LeftBot, *LeftTop, *RightBot, *RightTop;
    const int *TopLeft, *TopRight, *BotLeft, *BotRight;
    const double *xo, *yo;
} bgf_blocks;

/* Loop<T> time keeping (src/Arrays.h:358-366). */
typedef struct {
    double nextoutputtime;
    double dt;
    double dtmax;
    double totaltime;
} bgf_loop;

typedef struct bgf_handle_s* bgf_handle;

/* Last error message of the calling thread ("" if none). */
const char* bgf_last_error(void);

/* Library version string. */
const char* bgf_version(void);

/* Number of visible GPUs (0 without one). */
int bgf_device_count(void);

/* Allocates the device Model<T> for one domain on the current device and
 * uploads the block description.  Replaces AllocateGPU + CopytoGPU of
 * SetupGPU (src/Setup_GPU.cu:15-157). */
bgf_status bgf_create(const bgf_param* p, const bgf_blocks* b, bgf_handle* out);

/* Frees every device buffer of the handle. */
bgf_status bgf_destroy(bgf_handle h);

/* Uploads the state.  Arrays hold nblkmem*324 values of T (double for
 * BGF_FP64, float otherwise) in the reference layout; halo cells are ignored.
 * zb and cf are static: zb is the bed (Model.zb), cf the friction coefficient
 * (Model.cf).  zs is not an input: it is zb + h (src/Halo.cu:72-107). */
bgf_status bgf_set_state(bgf_handle h, const void* zb, const void* hh, const void* u, const void* v,
                         const void* cf);

/* Downloads zs, h, u, v (any pointer may be NULL) for the interior cells;
 * halo cells of the outputs are left untouched. */
bgf_status bgf_get_state(bgf_handle h, void* zs, void* hh, void* u, void* v);

/* Computes the first time step like initdt (src/Mainloop.cu:515-554):
 * loop->dtmax is set from dtinit (if > 0) and the per-cell
 * delta/sqrt(g*max(h,eps)) minimum, with the clamp of CalctimestepCPU. */
bgf_status bgf_init_dt(bgf_handle h, double dtinit, bgf_loop* loop);

/* One predictor-corrector step: FlowGPU<T>(XParam, XLoop, XForcing, XModel)
 * (src/FlowGPU.cu:14-315) with the CPU semantics of FlowCPU
 * (src/FlowCPU.cu:15-253).  Reads loop->totaltime, nextoutputtime and
 * dtmax; writes loop->dt and loop->dtmax like the reference.  The caller
 * advances totaltime (src/Mainloop.cu:60).  Synchronous. */
bgf_status bgf_step(bgf_handle h, bgf_loop* loop);

/* nsteps iterations of {bgf_step; totaltime += dt} that stay on the GPU
 * (device-resident loop state, no host round trip per step).  Steps stop
 * early, as no-ops, once totaltime >= endtime.  Returns the final loop. */
bgf_status bgf_run(bgf_handle h, bgf_loop* loop, int nsteps, double endtime);

/* Enqueues nsteps steps like bgf_run without waiting for them, on the
 * handle's stream.  bgf_sync waits and returns the loop state. */
bgf_status bgf_run_async(bgf_handle h, const bgf_loop* loop, int nsteps, double endtime);
bgf_status bgf_sync(bgf_handle h, bgf_loop* loop);

/* ---- the step on the caller's device Model<T> -------------------------------
 * MainLoop calls FlowGPU(XParam, XLoop, XForcing, XModel_g) with the device
 * copy of Model<T> (src/Mainloop.cu:51) and reads XModel_g's arrays right
 * after it (CrashDetection, Calcmeanmax, pointoutputstep, mapoutput:
 * src/Mainloop.cu:65-80).  These entry points take those device arrays
 * (nblkmem*324 values of the handle's T, the reference layout) as plain
 * device pointers. */

/* SetupGPU's upload when the caller's Model<T> is already on the device
 * (src/Setup_GPU.cu:15-157): copies zb, h, u, v, cf device-to-device. */
bgf_status bgf_set_state_device(bgf_handle h, const void* zb, const void* hh, const void* u, const void* v,
                                const void* cf);

/* FlowGPU<T>(XParam, XLoop, XForcing, XModel_g) (src/FlowGPU.cu:14-315) on
 * the caller's device arrays: one step from the state in hh, u, v (Model.evolv,
 * interior cells), written back into hh, zs (= zb + h), u, v (interior
 * cells) before the call returns, so the caller's post-step consumers see
 * U^{n+1} in XModel_g.evolv, as the reference's cleanup leaves it
 * (src/FlowGPU.cu:282).  zb: the bed if it changed since the last call
 * (deformstep), else NULL.  Loop semantics as bgf_step (writes dt and dtmax;
 * the caller advances totaltime).  Forcing as set on the handle
 * (bgf_set_rain_rate, bgf_set_rain_map_device, bgf_set_boundary,
 * bgf_set_rivers).  Synchronous. */
bgf_status bgf_step_device(bgf_handle h, void* hh, void* zs, void* u, void* v, const void* zb, bgf_loop* loop);

/* The one-level step that allocates nothing.  No counterpart in the
 * reference: it is for callers that cannot allocate device memory (code under
 * HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
 * One step as bgf_step (FlowGPU<T>, src/FlowGPU.cu:14-315; same kernels, same
 * results) of a one-level Cartesian domain held entirely in the caller's
 * device memory: d_blocks gives the block description as DEVICE arrays (active,
 * LeftBot, RightBot, BotLeft, TopLeft are read; they must describe a one-level
 * mesh, which is not checked), zb, cf, hh, u, v the state (nblkmem*324 values of
 * T, the reference layout), ho, uo, vo receive the new h, u, v of the interior
 * cells (distinct from the inputs).  loop as bgf_step (dt, dtmax written; the
 * caller advances totaltime).  Uniform rain from p->rain_on / p->rain; no other
 * forcing.  BGF_FP64, BGF_FP32 and BGF_FP32_FAST (BGF_FP32_COMP keeps per-cell
 * state across steps and needs a handle).  stream: a hipStream_t, or NULL;
 * the call waits for it.  The step's scratch (tendencies, block records, loop
 * state, work-queue counters) is one 64 MiB device array per GPU, held until
 * the process ends: at most 21,618 blocks (FP32 forms) or 10,865 blocks (FP64),
 * and as many block slots up to the greatest in the list (somewhat more where
 * the list is shorter), BGF_ERR_INVALID_ARG beyond.  Calls on one GPU share that array: calls that
 * overlap on one GPU (other threads, other streams) race. */
bgf_status bgf_step_noalloc(const bgf_param* p, const bgf_blocks* d_blocks, const void* zb, const void* cf,
                            const void* hh, const void* u, const void* v, void* ho, void* uo, void* vo,
                            bgf_loop* loop, void* stream);

/* Uniform rain rate [mm/h] of the coming steps: Forcing.Rain.nowvalue, which
 * updateforcing refreshes before each FlowGPU call (src/Updateforcing.cu:9-60,
 * src/Mainloop.cu:40).  Replaces the constant Param rate; a rate series or
 * map set on the handle takes precedence over it. */
bgf_status bgf_set_rain_rate(bgf_handle h, double rain_mmh);

/* The current rain map on the device: Forcing.Rain.now_g, nx*ny rates
 * [mm/h] row-major from (xo, yo) with spacing dx, which updateforcing
 * interpolates in time before each step.  The library reads it in place at
 * every step (the pointer must stay valid); NULL removes it. */
bgf_status bgf_set_rain_map_device(bgf_handle h, int nx, int ny, double xo, double yo, double dx,
                                   const float* now_g);

/* Copies n bytes of device memory to host memory, for callers that hold only
 * device Model<T> arrays (the block description at set-up). */
bgf_status bgf_copy_to_host(void* dst, const void* src, size_t n);

/* Gauges of a handle (the reference's point outputs, src/Mainloop.cu:359-500,
 * as batch members have them): up to 16 cells (memloc indices), whose depth
 * the GPU records after every `every`-th step counted from this call, up to
 * 2048 samples.  bgf_get_gauges copies values[g*2048 + k] (gauge g, sample k),
 * times[k] (totaltime after that step) and the sample count.  n = 0 removes
 * them, and so does bgf_remesh (the cells are indices of the old mesh). */
bgf_status bgf_set_gauges(bgf_handle h, int n, const int* cells, int every);
bgf_status bgf_get_gauges(bgf_handle h, float* values, double* times, int* nsamples);

/* Steps actually taken by the last bgf_run / bgf_run_async+bgf_sync (fewer
 * than asked when endtime was reached). */
bgf_status bgf_last_run_steps(bgf_handle h, int* nsteps);

/* Sum of h * delta^2 over active cells, accumulated in FP64 on the GPU. */
bgf_status bgf_volume(bgf_handle h, double* volume);

/* Device pointers of the handle's Model arrays by name ("h", "u", "v", "zb",
 * "cf", "dh", "dhu", "dhv"), for callers that keep Model<T> views.  The state
 * arrays use the block layout (324 values per block, halo included); on
 * one-level meshes the tendencies dh, dhu, dhv hold each block's 16x16
 * interior only (256 values per block, row y at 16*y) and live within a step. */
bgf_status bgf_device_array(bgf_handle h, const char* name, void** devptr);

/* Launch schedule of the persistent one-level kernels (no counterpart in the
 * reference, whose launches are one block per workgroup, src/FlowGPU.cu:14-315):
 * the active blocks are processed in tiles of tile_x x tile_y blocks, and the
 * predictor and corrector run wg_pred / wg_corr persistent workgroups per CU
 * (0 = as many as occupancy allows).  tile_x or tile_y 0 keeps the current
 * tile.  Results do not depend on the schedule; bg_flood_amd.autotune picks
 * one by timing.  Defaults: 16 x 12 blocks, occupancy; the environment
 * variable BGF_WG_PER_CU="p,c" sets the workgroups at creation. */
bgf_status bgf_set_schedule(bgf_handle h, int tile_x, int tile_y, int wg_pred, int wg_corr);
bgf_status bgf_get_schedule(bgf_handle h, int* tile_x, int* tile_y, int* wg_pred, int* wg_corr, int* grid_pred,
                            int* grid_corr);

/* Average duration, in milliseconds, of each kernel of the last bgf_run
 * call, measured with HIP events on the handle's stream when timing was
 * enabled with bgf_set_timing(h, 1).  names/ms receive up to n entries;
 * *count receives the number written. */
bgf_status bgf_set_timing(bgf_handle h, int enable);
bgf_status bgf_kernel_times(bgf_handle h, int n, const char** names, double* ms, int* count);

/* Builds the block list of a uniform one-level grid of nbx x nby blocks at
 * level `level`, in the raster order and with the neighbour convention of
 * InitBlockxoyo / InitBlockneighbours (src/Mesh.cu:257-433), in O(n).
 * xo/yo are computed in T (double if dbl, float otherwise) like the
 * reference and returned widened to double.  All arrays have nbx*nby
 * entries. */
bgf_status bgf_mesh_uniform(int nbx, int nby, double dx, int level, int dbl, int* active, int* lev,
                            double* xo, double* yo, int* LeftBot, int* LeftTop, int* RightBot,
                            int* RightTop, int* TopLeft, int* TopRight, int* BotLeft, int* BotRight);

/* Block list of a quadtree (multi-level) mesh from its leaves, with the
 * neighbour convention of the reference's adaptation
 * (src/Adaptation.cu:1017-1795; see bgf_blocks).  Leaf k becomes block k and
 * active[k] = k: level lev[k], integer block position (ix[k], iy[k]) among
 * the blocks of that level.  The domain is nbx x nby blocks at level `base`,
 * dx is the level-0 cell size.  The leaves must tile the domain and
 * neighbouring leaves may differ by one level at most (BGF_ERR_INVALID_ARG
 * otherwise).  Output arrays have nleaf entries. */
bgf_status bgf_mesh_from_leaves(int nleaf, const int* lev, const int* ix, const int* iy, int nbx, int nby, int base,
                                double dx, int* active, int* level, double* xo, double* yo, int* LeftBot,
                                int* LeftTop, int* RightBot, int* RightTop, int* TopLeft, int* TopRight,
                                int* BotLeft, int* BotRight);

/* One refinement pass of the quadtree with the reference's numbering
 * (src/Adaptation.cu:157-325 sanity cascade, 435-664 CalcAvailblk/AddBlocks,
 * 1017-1879 refine and cleanup; the reference cancels coarsening): blocks
 * whose refine_flags[ib] is set (and the coarser neighbours the 2:1 balance
 * forces) split in four; the block keeps its index as the bottom-left child
 * and the other three take free block slots in ascending order; new blocks
 * are appended to the active list.  p gives nblk, nblkmem, maxlevel, dx and
 * the precision the origins are stored in; b the current mesh (nbx x nby
 * level-0 blocks).  Outputs have `capacity` entries; *nblkmem_out may grow
 * (ceil((nblk + 3*nrefine) * 1.05)), BGF_ERR_OOM if it exceeds capacity.
 * Entries of unused slots: active -1, neighbours the slot itself. */
bgf_status bgf_adapt_refine(const bgf_param* p, const bgf_blocks* b, const unsigned char* refine_flags, int nbx,
                            int nby, int capacity, int* nblk_out, int* nblkmem_out, int* active, int* level,
                            double* xo, double* yo, int* LeftBot, int* LeftTop, int* RightBot, int* RightTop,
                            int* TopLeft, int* TopRight, int* BotLeft, int* BotRight);

/* Block description written by bgf_adapt_mesh (arrays of `capacity` entries). */
typedef struct {
    int* active;
    int* level;
    int *LeftBot, *LeftTop, *RightBot, *RightTop;
    int *TopLeft, *TopRight, *BotLeft, *BotRight;
    double *xo, *yo;
} bgf_blocks_out;

/* One adaptation pass with refinement and coarsening: Adapt's
 * refinesanitycheck, CalcAvailblk, AddBlocks, coarsen, refine and
 * Adaptationcleanup (src/Adaptation.cu:157-1876), with the reference's block
 * numbering.  coarsen_flags may be NULL: no coarsening, as the reference
 * itself (it cancels every coarsening request, :170-175).  With coarsen flags
 * the reference's coarsening rules apply: a block coarsens only as the
 * bottom-left of four same-level siblings that all request it, at a level
 * above minlevel, beside no finer block and no refining block.  remap (5 ints
 * per output slot, may be NULL) says where each slot's state comes from:
 * kind (-1 inactive, 0 kept, 1 child of a refined block, 2 coarsened parent)
 * then, for a child, its old parent and quadrant (0 BL, 1 BR, 2 TL, 3 TR),
 * for a coarsened parent its old BL, BR, TL, TR blocks, for a kept block its
 * own index.  Inputs and outputs as bgf_adapt_refine. */
bgf_status bgf_adapt_mesh(const bgf_param* p, const bgf_blocks* b, const unsigned char* refine_flags,
                          const unsigned char* coarsen_flags, int nbx, int nby, int capacity, int* nblk_out,
                          int* nblkmem_out, const bgf_blocks_out* out, int* remap);

/* Moves a multi-level handle's state onto the mesh of bgf_adapt_mesh, on the
 * GPU (the reference adapts on the CPU at set-up only, src/Adaptation.cu:17-
 * 155, and re-runs its initial conditions afterwards; this is the in-run
 * form).  p gives the new nblk and nblkmem (every other field as at
 * bgf_create).  Kept blocks keep their cells.  A child takes the bilinear
 * interpolation of its parent's h, zs, u, v (refine, :1032-1102) on the
 * parent's tile with its halo filled by the step's halo fill and corners by
 * fillCorners (src/Halo.cu:5277-5409); a coarsened parent the 2x2 means of
 * its children (coarsen, :700-760).  The bed of new cells comes from the bed
 * source of bgf_set_bed_source (interp2BUQ, src/GridManip.cu:333-560) when
 * one is set, else from the same interpolation of the old bed; then, on new
 * cells, h = max(eps, zs - zb) where h > eps and zs = zb elsewhere
 * (src/Adaptation.cu:493-512).  Roughness: a child cell takes its parent
 * cell's, a coarsened cell the mean.  The loop state (time, dt) is kept; the
 * next bgf_step or bgf_run continues on the new mesh. */
bgf_status bgf_remesh(bgf_handle h, const bgf_param* p, const bgf_blocks* b, const int* remap);

/* River discharges (the reference's rivers, src/Updateforcing.cu:146-363,
 * src/InitialConditions.cu:346-445): nriver rectangles boxes[4r..4r+3] =
 * (xstart, xend, ystart, yend) in the coordinates of Param.xo/yo, each with
 * a flow series of npts[r] (time [s], flow [m3/s]) pairs (times and flows
 * concatenated river by river).  A river discharges into the cells whose box
 * overlaps its rectangle, spread over their total area, added to the depth
 * tendency of both stages at the rate interpolated at the step's start.
 * Rivers that reach no cell are dropped, as in the reference; the discharge
 * cells are found again after bgf_remesh.  nriver = 0 removes them.
 * On spherical grids a cell's area is spharea (src/Spherical.cu:101-120) of its
 * centre and size in degrees, as the reference's set-up sums it
 * (src/InitialConditions.cu:385-388). */
bgf_status bgf_set_rivers(bgf_handle h, int nriver, const double* boxes, const int* npts, const double* times,
                          const double* flows);

/* Boundary segments (bndsegment, src/Forcing.h:106-150).  A segment has a type
 * (0 wall, noslipbndQ; 1 Neumann; 2 Dirichlet water level, Dirichlet1Q; 3
 * absorbing, ABS1DQ: bndFluxGPUSideCPU, src/Boundary.cu:587-741, 1887-2032; 4
 * accepted and acting as 1: the flux boundary of engine 2 has no branch for
 * it, src/Boundary.cu:688-726), a polygon, and a water level: a uniform series
 * of (time [s], level [m]) pairs interpolated at each stage's time
 * (src/Boundary.cu:116-145), a level map (below), or, without either,
 * Param.zsinit (0 when unset).  Every boundary block (one of its eight
 * neighbours is itself) belongs to the LAST segment whose polygon touches its
 * box (blockinpoly: a corner of the block inside the polygon or an edge
 * crossing), else to the remainder segment of type Param.aoibnd; all of a
 * block's boundary faces take its segment's type and level (Initbndblks,
 * src/InitialConditions.cu:1168-1290), so a corner block follows whichever of
 * its two sides' segments came later.  The assignment is redone on every new
 * mesh (bgf_remesh).  Not provided: atmospheric pressure at the boundary and
 * the absorbing boundary's mean flux filter (inactive unless Param.dt is set). */
#define BGF_MAX_SEGMENTS 64
typedef struct {
    int type;                 /* 0..4 */
    int side;                 /* 0 left, 1 right, 2 bottom, 3 top: the side's strip (readbndpolysegment,
                                 src/ReadForcing.cu:796-866, 2*dx wide); < 0: the polygon below */
    int npoly;                /* polygon vertices (>= 3), closed or not; made counter-clockwise */
    const double *px, *py;
    int nseries;              /* level series pairs (0, or >= 2 with increasing times) */
    const double *times, *levels;
} bgf_bnd_segment;

/* Replaces the segment list (the bndseg keys in file order, src/ReadInput.cu:919-962). */
bgf_status bgf_set_boundary_segments(bgf_handle h, int nseg, const bgf_bnd_segment* segs);

/* The segment of one side (the left/right/bot/top keys): replaces that side's
 * segment if there is one, else appends it.  Types 2 and 3 need a series of
 * n >= 2 pairs; other types take none. */
bgf_status bgf_set_boundary(bgf_handle h, int side, int type, int n, const double* times, const double* levels);

/* A level map for segment seg, making its level spatially varying (a boundary
 * given as a NetCDF file: WLmap, src/ReadInput.cu:1989-2001): nt frames of
 * nx*ny levels (x fastest; NaN read as 0, src/ReadForcing.cu:92) on the grid
 * from (xo, yo) by (dx, dy), at to + k*dt.  At each step's start the map is
 * interpolated between the frames bracketing totaltime (Forcingthisstep,
 * src/Updateforcing.cu:29-35, 54-127) and each boundary face samples it
 * bilinearly at its position (interp2BUQ, src/Boundary.cu:640-645). */
bgf_status bgf_set_boundary_map(bgf_handle h, int seg, int nx, int ny, double xo, double yo, double dx, double dy,
                                int nt, double to, double dt, const float* frames);

/* As bgf_set_boundary_map with the caller's current device map (WLmap.now_g,
 * kept current by the caller's Forcingthisstep), read in place each step;
 * NULL removes the map. */
bgf_status bgf_set_boundary_map_device(bgf_handle h, int seg, int nx, int ny, double xo, double yo, double dx,
                                       double dy, const float* now_g);

/* The segment of each block slot (nblkmem ints; -1: not a boundary block;
 * the remainder's index is the segment count). */
bgf_status bgf_boundary_blocks(bgf_handle h, int* out);

/* Param.zsoffset, Param.bndtaper, Param.inittime and Param.zsinit for the
 * boundaries (FlowbndFlux, src/Boundary.cu:108-195, bndFluxGPUSideCPU :648):
 * every level gains zsoffset (as a float, like the reference's zsbnd); with
 * bndtaper > 0 the level of a segment with a series or map ramps in from the
 * inside water level over bndtaper seconds after inittime (taper =
 * min((t - inittime) / bndtaper, 1) at the stage's time t); zsinit (NaN: unset,
 * 0) is the level of segments without either.  Defaults: 0, 0, 0, NaN. */
bgf_status bgf_set_boundary_options(bgf_handle h, double zsoffset, double bndtaper, double inittime, double zsinit);

/* Rain forcing beyond the constant Param rate (the Rain forcing of
 * src/Forcing.h:28-73, evaluated at the start of every step as updateforcing
 * does, src/Updateforcing.cu:9-127, then applied by the implicit rain of the
 * corrector, :530-581):
 *  - bgf_set_rain_series: a uniform rate as n >= 2 (time [s], rate [mm/h])
 *    pairs with increasing times, interpolated linearly in time (interptime);
 *    before the first and after the last pair the end segments extend;
 *  - bgf_set_rain_map: nframes frames of nx * ny rates [mm/h], row-major from
 *    (xo, yo) with spacing dx, at times t0 + k * dt; the map of a step is the
 *    linear interpolation between the frames that bracket its start
 *    (InterpstepCPU, src/GridManip.cu:602-622), sampled bilinearly at each
 *    cell centre (interp2BUQ).  One frame is a static map.
 * A map takes precedence over a series, a series over the constant rate.
 * n = 0 / nframes = 0 removes the forcing.  Handles only (batch members keep
 * their constant rates). */
bgf_status bgf_set_rain_series(bgf_handle h, int n, const double* times, const double* values);
bgf_status bgf_set_rain_map(bgf_handle h, int nx, int ny, double xo, double yo, double dx, int nframes, double t0,
                            double dt, const float* frames);

/* Bathymetry raster that bgf_remesh samples for new cells, as the reference
 * re-interpolates its bathymetry forcing after adaptation
 * (StaticForcingP<float>, src/Forcing.h): nx * ny values, row-major from
 * (xo, yo), spacing dx (and dy = dx), in the coordinates of Param.xo/yo.
 * NULL values removes it. */
bgf_status bgf_set_bed_source(bgf_handle h, int nx, int ny, double xo, double yo, double dx, const float* values);

/* Output statistics (Calcmeanmax, src/Meanmax.cu:15-112), updated on the GPU
 * after every step: mask 1 the means of h, zs, u, v (sums divided by the
 * step count at the step that reaches nextoutputtime) with U = |(u, v)|, h U
 * and h U U as the reference leaves them (assigned each step, then divided);
 * mask 2 the maxima of h, zs, u, v, U, h U, h U^2 (Param.outmax); mask 4 the
 * time each cell spent with h > wet_threshold (Param.outtwet).  zs = zb + h.
 * bgf_set_stats starts them (Initmeanmax: means and wet time 0, maxima
 * -max(T)); bgf_reset_stats resets those in `which` after an output
 * (resetmeanmax; the means also restart their step count); bgf_get_stats
 * copies one, by its output name ("hmean", "zsmean", "umean", "vmean",
 * "Umean", "hUmean", "hUUmean", "hmax", "zsmax", "umax", "vmax", "Umax",
 * "hUmax", "hUUmax", "twet"), as nblkmem*324 values of the handle's T.  A
 * remesh restarts them on the new mesh. */
bgf_status bgf_set_stats(bgf_handle h, int mask, double wet_threshold);
bgf_status bgf_reset_stats(bgf_handle h, int which);
bgf_status bgf_get_stats(bgf_handle h, const char* name, void* out);

/* A raster (values[i + j*nx] at xo + i*dx, yo + j*dx) sampled onto the
 * interior cells of the handle's mesh as interp2BUQ (src/GridManip.cu:333-560:
 * bilinear where the cell is no coarser than the raster, else the mean of the
 * raster points in the cell), into out (host, nblkmem*324 values of the
 * handle's T; other entries are left as they are).  Used for the hot start
 * (readhotstartfile, src/InitEvolv.cu:598-835) and for gridded inputs. */
bgf_status bgf_sample_raster(bgf_handle h, int nx, int ny, double xo, double yo, double dx, const float* values,
                             void* out);

/* Refinement flags of the reference's criteria on the GPU state
 * (src/AdaptCriteria.cu:62-160): per active block, mode 0 (Threshold) sets
 * flags[ib] if any interior cell of the field exceeds a; mode 1 (Inrange) if
 * any lies in [a, b]; mode 2 (steepness, no counterpart in the reference) if
 * the difference between two adjacent interior cells of the field, over the
 * block's cell size, exceeds a.  field: "h", "zs", "zb", "u" or "v".  flags
 * has nblkmem entries (0 for inactive blocks).  The reference's coarsening
 * flags are the complement of its refinement flags on the active blocks. */
bgf_status bgf_refine_flags(bgf_handle h, const char* field, int mode, double a, double b, unsigned char* flags);

/* ------------------------------------------------------------------ batches
 * A batch advances many independent domains ("members") with one
 * set of launches per step: ensembles, and continuous batching of solve
 * requests.  It has no counterpart in the reference, which runs one domain
 * per process (src/Mainloop.cu:17-91); each member follows FlowGPU<T>
 * semantics exactly as a bgf_handle would, with its own time step, time, end
 * time and rain rate.  Members are added and removed between runs; their
 * state stays on the GPU. */
typedef struct bgf_batch_s* bgf_batch;

/* Capacity: max_blocks block slots (a member takes its nblkmem) and
 * max_members members.  common gives the parameters shared by all members
 * (precision, g, eps, CFL, theta, delta, friction, boundary type, ...).
 * With common.maxlevel > common.minlevel the batch holds multi-level
 * (quadtree) members instead, whose block levels lie in that range and
 * whose dx and wetdryfix are common's: they are stepped by the multi-level
 * kernels (FP64, or FP32 in the reference's arithmetic for every FP32 form),
 * one set of launches for all of them, each block finding its member's loop
 * state; gauges, the running maximum depth, end times and membership changes
 * work as for one-level members. */
bgf_status bgf_batch_create(const bgf_param* common, int max_blocks, int max_members, bgf_batch* out);
bgf_status bgf_batch_destroy(bgf_batch b);

/* Adds a member: its own one-level block list (level 0) and state arrays
 * (nblkmem*324 values each, as bgf_set_state); p must match the batch's
 * common parameters except nblk, nblkmem and rain.  Its loop starts at
 * totaltime 0 with the initial step of initdt (src/Mainloop.cu:515-554;
 * dtinit <= 0 for the default) and lands exactly on endtime.  BGF_ERR_OOM
 * when the batch is full. */
bgf_status bgf_batch_add(bgf_batch b, const bgf_param* p, const bgf_blocks* blk, const void* zb, const void* hh,
                         const void* u, const void* v, const void* cf, double dtinit, double endtime, int* member);
bgf_status bgf_batch_remove(bgf_batch b, int member);

/* Enqueues nsteps batch steps: every member that has not reached its end
 * time takes one step of its own dt per batch step.  bgf_batch_sync waits. */
bgf_status bgf_batch_run_async(bgf_batch b, int nsteps);
bgf_status bgf_batch_sync(bgf_batch b);

/* Loop state of a member and whether it reached its end time. */
bgf_status bgf_batch_loop(bgf_batch b, int member, bgf_loop* loop, int* done);
/* Member state, as bgf_get_state. */
bgf_status bgf_batch_get_state(bgf_batch b, int member, void* zs, void* hh, void* u, void* v);
/* FP64 volume of a member, as bgf_volume. */
bgf_status bgf_batch_volume(bgf_batch b, int member, double* volume);

/* Output path (src/Meanmax.cu): folds the current depth of every member into
 * its running maximum (FP32, nblkmem*324 values per member); read it with
 * bgf_batch_get_maxdepth. */
bgf_status bgf_batch_update_maxdepth(bgf_batch b);
bgf_status bgf_batch_get_maxdepth(bgf_batch b, int member, float* hmax);

/* With tracking on, every step's corrector folds the depth into the running
 * maximum (instead of the snapshots of bgf_batch_update_maxdepth). */
bgf_status bgf_batch_track_maxdepth(bgf_batch b, int on);

/* Gauges: up to 16 cells (memloc indices in the member's arrays) per member,
 * recorded on the GPU after every `every`-th step of the member itself (so a
 * member's series do not depend on the rest of the batch), up to 2048
 * samples.  bgf_batch_get_gauges copies them: values[g*2048 + k] is gauge g
 * at sample k, times[k] its totaltime.  bgf_batch_sample_gauges reads the
 * current depth at every member's gauges now: 16*max_members values (NaN for
 * unused gauges) and, if times is not NULL, each member's totaltime. */
bgf_status bgf_batch_set_gauges(bgf_batch b, int member, int n, const int* cells, int every);
bgf_status bgf_batch_get_gauges(bgf_batch b, int member, float* values, double* times, int* nsamples);
bgf_status bgf_batch_sample_gauges(bgf_batch b, float* values, double* times);

/* Cell-updates performed so far, members and active blocks now. */
bgf_status bgf_batch_stats(bgf_batch b, long long* cell_updates, int* nmembers, int* nblocks);

/* Launch schedule of the batch's step, as bgf_set_schedule; a member's blocks
 * stay together and are tiled inside the member. */
bgf_status bgf_batch_set_schedule(bgf_batch b, int tile_x, int tile_y, int wg_pred, int wg_corr);
bgf_status bgf_batch_get_schedule(bgf_batch b, int* tile_x, int* tile_y, int* wg_pred, int* wg_corr);

/* ---- NetCDF files (no libnetcdf needed) ------------------------------------
 * BUQ map output as BG_Flood writes it (creatncfileBUQ, defncvarBUQ,
 * writencvarstepBUQ, writenctimestep: src/Write_netcdf.cu:118-500, 560-840,
 * 1215-1400), in the NetCDF classic format with 64-bit offsets (the reference
 * writes the same dimensions, variables and attributes into a NETCDF4 file).
 * The zone is the rectangle xo..xmax, yo..ymax of p (Param.xmax / ymax for
 * the whole domain, src/InitialConditions.cu:1105-1120) with levels
 * p->minlevel..p->maxlevel; every active block of b must lie in it.  names
 * are the output variables (Param.outvars); smallnc, scalefactor and
 * addoffset as Param.smallnc / scalefactor / addoffset. */
typedef struct bgf_ncout_s* bgf_ncout;
bgf_status bgf_nc_buq_create(const char* path, const bgf_param* p, const bgf_blocks* b, double xmax, double ymax,
                             int nvar, const char* const* names, int smallnc, float scalefactor, float addoffset,
                             bgf_ncout* out);
/* Appends one output (Save2Netcdf, src/Write_netcdf.cu:1703-1754): the time
 * and, for each variable, its host array in BUQ layout (nblkmem*324 values of
 * double when precision is BGF_FP64, else float). */
bgf_status bgf_nc_buq_write(bgf_ncout f, double time, int precision, const void* const* values);
bgf_status bgf_nc_buq_close(bgf_ncout f);

/* Reading NetCDF classic files (versions 1, 2 and 5; the reference reads any
 * NetCDF through libnetcdf, src/Read_netcdf.cu): a variable's shape (the
 * record dimension counts the records), its dimension names ("a,b,c"), one
 * record of a record variable (rec) or a whole fixed variable as doubles, and
 * a numeric attribute (var NULL or "" for a global one; n: capacity in,
 * count out). */
bgf_status bgf_nc_inq(const char* path, const char* var, int* ndim, long long* shape, int* is_record);
bgf_status bgf_nc_dim_names(const char* path, const char* var, char* names, int cap);
bgf_status bgf_nc_get(const char* path, const char* var, long long rec, double* out);
bgf_status bgf_nc_get_att(const char* path, const char* var, const char* att, double* out, int* n);

#ifdef __cplusplus
}
#endif
#endif
