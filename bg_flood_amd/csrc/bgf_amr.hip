// bgf_amr.hip -- the Kurganov step on multi-level (quadtree) block meshes.
//
// On a mesh whose blocks differ in level the halo of a block is no longer a
// copy of its neighbours' edge cells: it is a restriction (2x2 mean of a finer
// neighbour), a barycentric prolongation from a coarser neighbour, a linear
// reconstruction from the coarse gradients, and the coarse face fluxes are the
// means of the fine ones.  Blocks keep the reference's Model<T> layout (18x18
// tiles).  Per step:
//
//   k_amr_stage      predictor: the block's halo of h, u, v
//                    (src/Halo.cu:2083-4609) with the wet/dry restriction of h
//                    (src/ConserveElevation.cu:218-378,676-726), and beside a
//                    coarser block the linear prolongation
//                    (src/Halo.cu:1044-1405), whose coarse theta-minmod slopes
//                    (src/Gradients.cu:921-957: of the reference's first
//                    gradient pass only these are read) are formed from the
//                    cells the coarse block's fill reads, and the wet/dry
//                    prolongation (src/ConserveElevation.cu:80-205, 451-482);
//                    then the gradients with their halo values
//                    (src/Gradients.cu:2584-3294), the faces
//                    (src/Kurganov.cu:474-641, 1404-1546) with the coarse-face
//                    source substitution, and the tendencies
//                    (src/Advection.cu:160-254), all in LDS; zs = zb + h
//                    (src/Halo.cu:72-107) is formed where it is read.  The
//                    block's largest wave speed goes to the dt slots.
//   k_amr_advance    the dt reduction and U* = U + dt/2 L(U)
//                    (src/Advection.cu:332-385).  A block beside a finer one
//                    takes its shared faces as the means of the finer faces
//                    first (src/Halo.cu:1441-1862), a block on an open
//                    boundary the boundary's (src/Boundary.cu:587-760).
//   k_amr_stage      corrector: the same on U*, and then the advance with
//                    bottom friction, cleanup and implicit rain, except
//   k_amr_fix_advance  in the blocks beside finer ones, or on open boundaries,
//                    which wait for the others' faces.
//
// The step used to run as halo, prolongation, gradients and fluxes, and
// fix-up and advance, two of each, with eight face arrays between them: 103 us
// a step on a mesh of 1,607 blocks in FP32 and 2.01 ms on 39,348 blocks in
// FP64; with the stage in one launch and faces stored only where another
// block reads them 66 us and 0.98 ms; with the mesh's gather recipes formed
// beforehand (k_amr_recipes) 48 us and 0.94 ms.
//
// On meshes of four levels and more the halos are filled by a launch of their
// own (k_amr_halo_refine) and prolonged level by level (k_amr_prolong).
//
// Threads map to halo cells by (side, j): side 0 left, 1 right, 2 bottom,
// 3 top, j the position along the side.  Every formula keeps the reference
// CPU step's operation order and precision (this file is built with
// -ffp-contract=off), including the per-side differences of the reference:
// the order of the four terms of the gradient-halo means, the argument order
// of the bilinear interpolation, and refine_linear's double-precision
// ilevdx on the left and top sides.
//
// Sequential order.  The reference visits blocks in active-list order, and in
// the wet/dry prolongation a block's test reads the halo of its coarser
// neighbour, which that neighbour's own prolongation may already have
// rewritten: it sees the prolonged value if that neighbour comes earlier in
// the active list.  Only a halo cell of the coarser block beside a still
// coarser one is ever rewritten, so with three levels the chain ends there and
// a block evaluates that cell again (the EH_* cells of k_amr_stage).  The bed
// of such a halo cell may be written by the coarser block's workgroup in the
// same launch, but only with the bed of the cell that the evaluation takes
// instead, so what was read of it is not used.  Every other stage only reads
// cells that the same launch does not write, so blocks run in parallel.

#include <hip/hip_runtime.h>

#include <cfloat>

#include "bgf_common.h"

namespace bgf {
namespace {

enum { SL = 0, SR = 1, SB = 2, ST = 3 };

template <class T> __device__ __forceinline__ T epsi_of() {
    return sizeof(T) == 8 ? T(2.220446049250313e-16) : T(1.1920928955078125e-07);
}
template <class T> __device__ __forceinline__ T tmax_of() { return sizeof(T) == 8 ? T(DBL_MAX) : T(FLT_MAX); }

// std::max / std::min with their NaN and signed-zero behaviour.
template <class T> __device__ __forceinline__ T smax(T a, T b) { return (a < b) ? b : a; }
template <class T> __device__ __forceinline__ T smin(T a, T b) { return (b < a) ? b : a; }

// src/Util_CPU.cu:308-311
template <class T> __device__ __forceinline__ int ftoi(T v) {
    return v >= T(0) ? (int)(v + T(0.5)) : (int)(v - T(0.5));
}

// A side of a block: the neighbours covering its first half (bottom or left)
// and second half (top or right), itself at the domain edge; their levels;
// and, beside a coarser neighbour, whether the block is that neighbour's
// first-half neighbour.  Read from the block's record nbr (sides in the order
// left, right, bottom, top, first and second half each, then the same places
// for the levels and flags): one record instead of a selection among the
// eight neighbour arrays, which would index the parameter struct by a
// per-thread side and put it in scratch memory.
struct Side {
    int n1, n2, l1, l2;
    bool back;
};
__device__ __forceinline__ int rec_level(int info) { return (int)(signed char)(info & 0xff); }
__device__ __forceinline__ Side make_side(int n1, int n2, int i1, int i2) {
    return Side{n1, n2, rec_level(i1), rec_level(i2), ((i1 & REC_BACK) != 0)};
}
__device__ __forceinline__ Side side_of(const KParams& P, int s, int b) {
    const int2 n = *(const int2*)(P.nbr + b * NBR + 2 * s), i = *(const int2*)(P.nbr + b * NBR + 8 + 2 * s);
    return make_side(n.x, n.y, i.x, i.y);
}
// The same where s and b are uniform over the wave, in scalar loads.
__device__ __forceinline__ Side side_of_uniform(const KParams& P, int s, int b) {
    const int o = b * NBR + 2 * s;
    return make_side(ldu(P.nbr, o), ldu(P.nbr, o + 1), ldu(P.nbr, o + 8), ldu(P.nbr, o + 9));
}
// Neighbours of a coarser block C next to the ends of the shared side: before
// its first cell (j == 0) and after its last (j == 15), on the half facing us;
// lev receives their level.
__device__ __forceinline__ int corner_lo(const KParams& P, int s, int C, int& lev) {
    const Side S = side_of(P, s < 2 ? SB : SL, C);
    const bool second = s == SL || s == SB;
    lev = second ? S.l2 : S.l1;
    return second ? S.n2 : S.n1;
}
__device__ __forceinline__ int corner_hi(const KParams& P, int s, int C, int& lev) {
    const Side S = side_of(P, s < 2 ? ST : SR, C);
    const bool second = s == SL || s == SB;
    lev = second ? S.l2 : S.l1;
    return second ? S.n2 : S.n1;
}
// Cell at depth d from side s of block b, at position k along the side
// (d = -1 is the halo cell).
__device__ __forceinline__ int edge_cell(int s, int d, int k, int b) {
    return s == SL ? memloc(d, k, b) : s == SR ? memloc(BW - 1 - d, k, b) : s == SB ? memloc(k, d, b)
                                                                                   : memloc(k, BW - 1 - d, b);
}

// A field value: the array itself, or zs = zb + h.
template <class T, bool ZS> struct Fld {
    const T* a;
    const T* zb;
    __device__ __forceinline__ T operator()(int c) const { return ZS ? zb[c] + a[c] : a[c]; }
};

// ---------------------------------------------------------------- gathers
// A halo value is a fixed combination of up to four cells of the Model arrays.
// Its recipe (which cells, which formula) depends on the mesh only; the
// kernels form every recipe a thread needs first, then load all their cells,
// then combine, so that the loads of one thread are in flight together
// instead of one dependent wait per branch.
enum { G_COPY = 0, G_MEAN4 = 1, G_W3 = 2, G_BILIN = 3 };
template <class T> struct Gather {
    int kind;
    int i[4];  // cells; unused places repeat i[0]
    T a, b, c; // G_W3: the weights of i[0..2]; G_BILIN: the point (a, b)
    int set;   // G_W3: which weights (w3_weights)
};
template <class T> __device__ __forceinline__ Gather<T> g_copy(int c) {
    return Gather<T>{G_COPY, {c, c, c, c}, T(0), T(0), T(0), 0};
}
template <class T> __device__ __forceinline__ Gather<T> g_mean4(int c0, int c1, int c2, int c3) {
    return Gather<T>{G_MEAN4, {c0, c1, c2, c3}, T(0), T(0), T(0), 0};
}
// The weights of a halo cell beside a coarser block: of the own edge cell and
// of the coarse cells after and before it (src/Halo.cu:2083-2286): W3_UP, W3_DOWN
// the nearer one counts more; at the end of a side, by the block beside the
// coarse one: W3_SAME none, W3_AFTER and W3_BEFORE a coarser one (beyond the
// side's first and last cell), W3_FINE a finer one.
enum { W3_UP = 0, W3_DOWN = 1, W3_SAME = 2, W3_AFTER = 3, W3_BEFORE = 4, W3_FINE = 5 };
template <class T> __device__ __forceinline__ void w3_weights(int set, T& a, T& b, T& c) {
    a = T(1.0 / 3.0);
    // T(0.5*(1.0-w1)) and T(0.5)*(T(1.0)-w1) round to the same float
    const T half = T(0.5 * (1.0 - (double)T(1.0 / 3.0)));
    b = set == W3_UP ? T(1.0 / 6.0) : set == W3_SAME ? half : T(0.5);
    c = set == W3_UP ? T(0.5) : set == W3_SAME ? half : T(1.0 / 6.0);
    if (set == W3_AFTER) { a = T(4.0 / 10.0); b = T(5.0 / 10.0); c = T(1.0 / 10.0); }
    if (set == W3_BEFORE) { a = T(4.0 / 10.0); b = T(1.0 / 10.0); c = T(5.0 / 10.0); }
    if (set == W3_FINE) { a = T(1.0 / 4.0); b = T(1.0 / 2.0); c = T(1.0 / 4.0); }
}

// src/Util_CPU.cu:129-144 on the unit square.
template <class T> __device__ __forceinline__ T bilinear(T q11, T q12, T q21, T q22, T x, T y) {
    const T x1 = T(0.0), x2 = T(1.0), y1 = T(0.0), y2 = T(1.0);
    const T x2x1 = x2 - x1, y2y1 = y2 - y1, x2x = x2 - x, y2y = y2 - y, yy1 = y - y1, xx1 = x - x1;
    return T(1.0) / (x2x1 * y2y1) * (q11 * x2x * y2y + q21 * xx1 * y2y + q12 * x2x * yy1 + q22 * xx1 * yy1);
}

// The combination of the recipe's cell values z[0..3] (loaded in its order).
template <class T> __device__ __forceinline__ T g_apply(const Gather<T>& g, const T* z) {
    switch (g.kind) {
        case G_COPY: return z[0];
        case G_MEAN4: return T(0.25) * (z[0] + z[1] + z[2] + z[3]);
        case G_W3: return g.a * z[0] + g.b * z[1] + g.c * z[2];
        default: return bilinear(z[0], z[1], z[2], z[3], g.a, g.b);
    }
}
template <class T> __device__ __forceinline__ void g_load(const Gather<T>& g, const T* a, T* z) {
#pragma unroll
    for (int m = 0; m < 4; m++) z[m] = a[g.i[m]];
}

// ------------------------------------------------------------- halo fill
// 2x2 mean of a finer neighbour's cells next to the shared edge.
template <class T> __device__ __forceinline__ Gather<T> mean_fine(int os, int n, int jj) {
    return g_mean4<T>(edge_cell(os, 0, jj, n), edge_cell(os, 1, jj, n), edge_cell(os, 0, jj + 1, n),
                      edge_cell(os, 1, jj + 1, n));
}

// Halo value of side s, position j (src/Halo.cu:2083-2286 and its three mirrors).
// S: side s of block ib; lev: the level of block ib.
template <class T>
__device__ __forceinline__ Gather<T> fill_recipe(const KParams& P, const Side& S, int s, int j, int ib, int lev) {
    const int os = s ^ 1;
    const int n1 = S.n1, n2 = S.n2;
    if (n1 == ib) {
        if (j < BW / 2 || n2 == ib) return g_copy<T>(edge_cell(s, 0, j, ib));
        return mean_fine<T>(os, n2, (j - BW / 2) * 2);
    }
    const int l1 = S.l1;
    if (l1 == lev) return g_copy<T>(edge_cell(os, 0, j, n1));
    if (l1 > lev) {
        if (j < BW / 2) return mean_fine<T>(os, n1, j * 2);
        if (n2 == ib) return g_copy<T>(edge_cell(s, 0, j, ib));
        return mean_fine<T>(os, n2, (j - BW / 2) * 2);
    }
    // coarser neighbour: 1/3 own edge cell + {1/6, 1/2} of the two nearest coarse cells
    const int C = n1;
    const bool first = S.back;
    const T cj = ceil(T(j) * T(0.5));
    const int jjc = first ? ftoi(cj) : ftoi(cj + T(BW / 2));
    const bool up = cj * T(2) > T(j);
    int set = up ? W3_UP : W3_DOWN;
    const int ii = edge_cell(s, 0, j, ib);
    int ir = edge_cell(os, 0, jjc, C);
    int it = edge_cell(os, 0, jjc - 1, C);
    if (first) {
        if (j == 0) {
            int ln;
            const int n = corner_lo(P, s, C, ln);
            if (n == C) {
                set = W3_SAME;
                it = ir;
            } else {
                it = edge_cell(os, 0, BW - 1, n);
                if (ln < l1) set = W3_AFTER;
                else if (ln > l1) set = W3_FINE;
            }
        }
    } else if (j == BW - 1) {
        const int C2 = S.n2, l2 = S.l2;
        int ln;
        const int n = corner_hi(P, s, C2, ln);
        if (n == C2) {
            set = W3_SAME;
            ir = it;
        } else {
            ir = edge_cell(os, 0, 0, n);
            if (ln < l2) set = W3_BEFORE;
            else if (ln > l2) set = W3_FINE;
        }
    }
    Gather<T> g{G_W3, {ii, ir, it, ii}, T(0), T(0), T(0), set};
    w3_weights(set, g.a, g.b, g.c);
    return g;
}
template <class T> __device__ __forceinline__ T fill_value(const KParams& P, int s, int j, int ib, const T* z) {
    const Gather<T> g = fill_recipe<T>(P, side_of(P, s, ib), s, j, ib, P.level[ib]);
    T zz[4];
    g_load(g, z, zz);
    return g_apply(g, zz);
}

// Wet/dry restriction of one coarse halo cell beside a finer block
// (src/ConserveElevation.cu:676-726): on when the option is set and the
// neighbour on that half of side s is finer; the 2x2 fine patch's cells
// (lower-left, right, top, top-right) and the halo cell itself (its bed).
struct WetDry {
    int on;
    int i[4];
    int w;
};
__device__ __forceinline__ WetDry wetdry_recipe(const KParams& P, const Side& S, int s, int j, int ib, int lev) {
    WetDry r;
    const int n = j < BW / 2 ? S.n1 : S.n2;
    r.on = P.wetdryfix && lev < (j < BW / 2 ? S.l1 : S.l2);
    const int jr = (j & (BW / 2 - 1)) * 2;
    const int i0 = s == SL ? BW - 2 : s == SR ? 0 : jr;
    const int j0 = s == SB ? BW - 2 : s == ST ? 0 : jr;
    r.i[0] = memloc(i0, j0, n);
    r.i[1] = memloc(i0 + 1, j0, n);
    r.i[2] = memloc(i0, j0 + 1, n);
    r.i[3] = memloc(i0 + 1, j0 + 1, n);
    r.w = edge_cell(s, -1, j, ib);
    return r;
}
// The restricted depth from the patch's h and zb (hh, zz in the recipe's
// order) and the halo cell's bed zbw, or hv, the filled depth, where the patch
// is all wet or all dry.
template <class T> __device__ __forceinline__ T wetdry_apply(T eps, const T* hh, const T* zz, T zbw, T hv) {
    const T iiwet = hh[0] > eps ? T(1.0) : T(0.0);
    const T irwet = hh[1] > eps ? T(1.0) : T(0.0);
    const T itwet = hh[2] > eps ? T(1.0) : T(0.0);
    const T itrwet = hh[3] > eps ? T(1.0) : T(0.0);
    const T cwet = iiwet + irwet + itwet + itrwet;
    T hwet = iiwet * hh[0] + irwet * hh[1] + itwet * hh[2] + itrwet * hh[3];
    T zswet = (iiwet * hh[0]) * (zz[0] + hh[0]) + (irwet * hh[1]) * (zz[1] + hh[1]) +
              (itwet * hh[2]) * (zz[2] + hh[2]) + (itrwet * hh[3]) * (zz[3] + hh[3]);
    if (cwet > T(0.0) && cwet < T(4.0)) {
        zswet = zswet / hwet;
        return smax(T(0.0), zswet - zbw);
    }
    return hv;
}

// Four blocks per workgroup, 64 threads per block: (side, j) = (t/16 % 4, t % 16).
// vb is the work unit (a workgroup index of a launch over quads of blocks).
__device__ __forceinline__ int quad_block(const KParams& P, int t, int vb) {
    const int ibl = vb * 4 + (t >> 6);
    return ibl < P.nblk ? P.active[ibl] : -1;
}

// The loop state of block ib: its member's in a batch of domains (P.sid), else
// the one loop state.
__device__ __forceinline__ DevLoop* loop_of(const KParams& P, DevLoop* L, int ib) {
    return P.sid ? L + P.sid[ib] : L;
}
// Whether the stage of block ib's domain is skipped: the predictor's once the
// domain reached its end time, the corrector's when the reduction did not start it.
__device__ __forceinline__ bool stage_off(const DevLoop* L, int corr) { return corr ? !L->go : L->done; }

// The depth the halo fill gives halo cell (s, j) of block ib: the fill, or
// beside a finer block the wet/dry restriction where it applies.
template <class T>
__device__ __forceinline__ T halo_depth(const KParams& P, const T* h, const T* zb, int s, int j, int ib) {
    const int lev = P.level[ib];
    T hv = fill_value(P, s, j, ib, h);
    const WetDry wd = wetdry_recipe(P, side_of(P, s, ib), s, j, ib, lev);
    if (wd.on) {
        T hh[4], zz[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            hh[m] = h[wd.i[m]];
            zz[m] = zb[wd.i[m]];
        }
        hv = wetdry_apply(T(P.eps), hh, zz, zb[wd.w], hv);
    }
    return hv;
}

// The halo cell (s, j) of block ib.
template <class T>
__device__ __forceinline__ void amr_halo_side(const KParams& P, T* h, T* u, T* v, const T* zb, int s, int j, int ib) {
    const int w = edge_cell(s, -1, j, ib);
    const T hv = halo_depth(P, h, zb, s, j, ib);
    const T uv = fill_value(P, s, j, ib, u);
    const T vv = fill_value(P, s, j, ib, v);
    h[w] = hv;
    u[w] = uv;
    v[w] = vv;
}
template <class T>
__global__ __launch_bounds__(256) void k_amr_halo(KParams P, T* h, T* u, T* v, const T* zb) {
    const int t = threadIdx.x, ib = quad_block(P, t, blockIdx.x);
    if (ib >= 0) amr_halo_side<T>(P, h, u, v, zb, (t >> 4) & 3, t & 15, ib);
}

// Halo of one static field (the bed at set-up, src/InitialConditions.cu:135-147).
template <class T> __global__ __launch_bounds__(256) void k_amr_fill(KParams P, T* z) {
    const int t = threadIdx.x;
    const int ib = quad_block(P, t, blockIdx.x);
    if (ib < 0) return;
    const int s = (t >> 4) & 3, j = t & 15;
    z[edge_cell(s, -1, j, ib)] = fill_value(P, s, j, ib, z);
}

// ------------------------------------------------------------- gradients
// src/Util_CPU.cu:243-263
template <class T> __device__ __forceinline__ T minmod2(T theta, T s0, T s1, T s2) {
    if (s0 < s1 && s1 < s2) {
        T d1 = theta * (s1 - s0);
        const T d2 = (s2 - s0) / T(2.0);
        const T d3 = theta * (s2 - s1);
        if (d2 < d1) d1 = d2;
        return smin(d1, d3);
    }
    if (s0 > s1 && s1 > s2) {
        T d1 = theta * (s1 - s0);
        const T d2 = (s2 - s0) / T(2.0);
        const T d3 = theta * (s2 - s1);
        if (d2 > d1) d1 = d2;
        return smax(d1, d3);
    }
    return T(0.0);
}

// Value two cells beyond the edge on side s, the outer point of the limited
// gradient at the halo cell (src/Gradients.cu:2713-3294); lev: block ib's level.
template <class T> __device__ __forceinline__ Gather<T> far_recipe(const Side& S, int s, int j, int ib, int lev) {
    const int os = s ^ 1;
    const int n1 = S.n1, n2 = S.n2;
    // finer neighbour: mean of its depth-2 and depth-3 cells; the left and
    // bottom sides add the depth-2 cell first, the right and top sides the depth-3 cell
    const int da = (s == SL || s == SB) ? 2 : 3, db = 5 - da;
    auto mean2 = [&](int n, int jj) {
        return g_mean4<T>(edge_cell(os, da, jj, n), edge_cell(os, db, jj, n), edge_cell(os, da, jj + 1, n),
                          edge_cell(os, db, jj + 1, n));
    };
    if (n1 == ib) {
        if (j < BW / 2 || n2 == ib) return g_copy<T>(edge_cell(s, 0, j, ib));
        return mean2(n2, (j - BW / 2) * 2);
    }
    const int l1 = S.l1;
    if (l1 == lev) return g_copy<T>(edge_cell(os, 1, j, n1));
    if (l1 > lev) {
        if (j < BW / 2) return mean2(n1, j * 2);
        if (n2 == ib) return g_copy<T>(edge_cell(s, 0, j, ib));
        return mean2(n2, (j - BW / 2) * 2);
    }
    const int C = n1;
    const T cj = ceil(T(j) * T(0.5));
    const int jj = S.back ? ftoi(cj) : ftoi(cj + T(BW / 2));
    const T jr = cj * T(2) > T(j) ? T(0.25) : T(0.75);
    const int p0 = edge_cell(os, 0, jj, C), p1 = edge_cell(os, 1, jj, C);
    const int q0 = edge_cell(os, 0, jj - 1, C), q1 = edge_cell(os, 1, jj - 1, C);
    // bilinear(q11, q12, q21, q22, x, y) with the side's corner order
    switch (s) {
        case SL: return Gather<T>{G_BILIN, {q1, p1, q0, p0}, T(0.75), jr, T(0), 0};
        case SR: return Gather<T>{G_BILIN, {q0, p0, q1, p1}, T(0.25), jr, T(0), 0};
        case SB: return Gather<T>{G_BILIN, {q1, q0, p1, p0}, jr, T(0.75), T(0), 0};
        default: return Gather<T>{G_BILIN, {q0, q1, p0, p1}, jr, T(0.25), T(0), 0};
    }
}

// ----------------------------------------------------------- prolongation
// Cell (x, y) of block C, x, y in [-1, 16] with at most one of them outside
// [0, 15], as a gather: the cell itself, or C's halo cell as the fill leaves
// it (for h with the wet/dry restriction); levC: C's level.
template <class T> struct HaloPt {
    Gather<T> g;
    WetDry wd;
};
template <class T> __device__ __forceinline__ HaloPt<T> pt_recipe(const KParams& P, int x, int y, int C, int levC) {
    HaloPt<T> r;
    if (x >= 0 && x < BW && y >= 0 && y < BW) {
        const int c = memloc(x, y, C);
        r.g = g_copy<T>(c);
        r.wd = WetDry{0, {c, c, c, c}, c};
        return r;
    }
    const int s = x < 0 ? SL : x >= BW ? SR : y < 0 ? SB : ST;
    const int j = s < 2 ? y : x;
    const Side S = side_of(P, s, C);
    r.g = fill_recipe<T>(P, S, s, j, C, levC);
    r.wd = wetdry_recipe(P, S, s, j, C, levC);
    return r;
}

// Linear reconstruction z_c + (+-dzdx_c +- dzdy_c) * dx_f / 2 of halo cell
// (s, j) of a block of level lev beside the coarser block C (src/Halo.cu:
// 1044-1066 and mirrors) from z at C's edge cell c and its four neighbours
// f[0..4] = (c, x-1, x+1, y-1, y+1).  The coarse slopes are those of the
// gradient pass that runs before it (src/Gradients.cu:921-957): theta-minmod
// of C's cells and of its halo as the fill leaves it, here formed from the
// cells the fill reads (no block's halo is read while another block writes
// its own).
template <class T>
__device__ __forceinline__ T refine_from(const KParams& P, int s, int j, int lev, int levC, const T* f) {
    const T theta = T(P.theta);
    const T dc = calcres(T(P.delta0), levC);
    const T zc = f[0];
    const T dzdx = minmod2(theta, f[1], zc, f[2]) / dc;
    const T dzdy = minmod2(theta, f[3], zc, f[4]) / dc;
    const T fj = floor(T(j) * T(0.5));
    const T along = fj * T(2.0) < (T(j) - T(0.01)) ? T(1.0) : T(-1.0);
    const T nrm = (s == SL || s == SB) ? T(1.0) : T(-1.0);
    const T faclr = s < 2 ? nrm : along, facbt = s < 2 ? along : nrm;
    const T slope = faclr * dzdx + facbt * dzdy;
    if (s == SL || s == ST) {
        const double ilevdx = calcres(P.delta0, lev) * (double)T(0.5);
        return T((double)zc + (double)slope * ilevdx);
    }
    const T ilevdx = calcres(T(P.delta0), lev) * T(0.5);
    return zc + slope * ilevdx;
}

// Halo cell (s, j) of block ib (level lev) for a stage: the fill
// (src/Halo.cu:2083-4609) with the wet/dry restriction
// (src/ConserveElevation.cu:676-726), or beside a coarser block the linear
// reconstruction; hs keeps h as it then stands for the prolongation.  Beside
// a coarser block C on the coarsest level, the wet/dry prolongation
// (src/ConserveElevation.cu:80-205) follows at once: C has no coarser
// neighbour, so its halo is the fill whatever the order of the reference's
// sequential pass; the finer levels take k_amr_prolong.  The recipes of all
// points come first, then every load, then the arithmetic.
template <class T> struct HaloVals {
    T h, u, v;  // the halo cell's values
    T hs;       // h before the wet/dry prolongation
    T zb;       // the bed the prolongation gives it (zbset)
    bool zbset;
};
template <class T>
__device__ __forceinline__ HaloVals<T> amr_halo_refine(const KParams& P, const T* h, const T* u, const T* v,
                                                       const T* zb, bool prolong, int s, int j, int ib, int lev) {
    const Side S = side_of(P, s, ib);
    const int C = S.n1, levC = S.l1;
    const bool coarse = levC < lev;
    const bool pro = coarse && prolong && levC == P.minlevel;
    HaloPt<T> pt[5];
    if (coarse) {
        const T fj = floor(T(j) * T(0.5));
        const int jj = S.back ? ftoi(fj) : ftoi(fj + T(BW / 2));
        const int cx = s == SL ? BW - 1 : s == SR ? 0 : jj, cy = s == SB ? BW - 1 : s == ST ? 0 : jj;
        pt[0] = pt_recipe<T>(P, cx, cy, C, levC);
        pt[1] = pt_recipe<T>(P, cx - 1, cy, C, levC);
        pt[2] = pt_recipe<T>(P, cx + 1, cy, C, levC);
        pt[3] = pt_recipe<T>(P, cx, cy - 1, C, levC);
        pt[4] = pt_recipe<T>(P, cx, cy + 1, C, levC);
    } else {
        pt[0].g = fill_recipe<T>(P, S, s, j, ib, lev);
        pt[0].wd = wetdry_recipe(P, S, s, j, ib, lev);
#pragma unroll
        for (int k = 1; k < 5; k++) pt[k].wd.on = 0;
    }
    T H[5][4], U[5][4], V[5][4], WH[5][4], WZ[5][4], WZW[5];
    g_load(pt[0].g, h, H[0]);
    g_load(pt[0].g, u, U[0]);
    g_load(pt[0].g, v, V[0]);
    if (coarse) {
#pragma unroll
        for (int k = 1; k < 5; k++) {
            g_load(pt[k].g, h, H[k]);
            g_load(pt[k].g, u, U[k]);
            g_load(pt[k].g, v, V[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < 5; k++) {
        if (pt[k].wd.on) {
#pragma unroll
            for (int m = 0; m < 4; m++) {
                WH[k][m] = h[pt[k].wd.i[m]];
                WZ[k][m] = zb[pt[k].wd.i[m]];
            }
            WZW[k] = zb[pt[k].wd.w];
        }
    }
    const T zbc = pro ? zb[pt[0].g.i[0]] : T(0);
    const T eps = T(P.eps);
    T hv[5], uv[5], vv[5];
#pragma unroll
    for (int k = 0; k < 5; k++) {
        if (k > 0 && !coarse) break;
        hv[k] = g_apply(pt[k].g, H[k]);
        if (pt[k].wd.on) hv[k] = wetdry_apply(eps, WH[k], WZ[k], WZW[k], hv[k]);
        uv[k] = g_apply(pt[k].g, U[k]);
        vv[k] = g_apply(pt[k].g, V[k]);
    }
    HaloVals<T> o;
    o.zbset = false;
    if (!coarse) {
        o.h = hv[0];
        o.u = uv[0];
        o.v = vv[0];
        o.hs = o.h;
        return o;
    }
    o.h = refine_from(P, s, j, lev, levC, hv);
    o.u = refine_from(P, s, j, lev, levC, uv);
    o.v = refine_from(P, s, j, lev, levC, vv);
    o.hs = o.h;
    if (pro && !(hv[0] > eps && hv[1] > eps && hv[2] > eps && hv[4] > eps && hv[3] > eps)) {
        o.h = hv[0];
        o.zb = zbc;
        o.zbset = true;
    }
    return o;
}

// Wet/dry prolongation of the blocks of one level (src/ConserveElevation.cu:80-205):
// where the coarse cell or one of its four neighbours is dry, the halo takes
// the coarse cell's h and zb.
template <class T>
__device__ __forceinline__ void amr_prolong(const KParams& P, T* h, T* zb, const T* hsnap, int level, DevLoop* L,
                                            int corr, int t, int vb) {
    const int ib = quad_block(P, t, vb);
    if (ib < 0) return;
    const int lev = P.level[ib];
    if (lev != level) return;
    const int s = (t >> 4) & 3, j = t & 15;
    const Side S = side_of(P, s, ib);
    const int C = S.n1;
    if (!(lev > S.l1)) return;
    const T eps = T(P.eps);
    const T fj = floor(T(j) * T(0.5));
    const int jp = S.back ? ftoi(fj) : ftoi(fj + T(BW / 2));
    const int cx = s == SL ? BW - 1 : s == SR ? 0 : jp;
    const int cy = s == SB ? BW - 1 : s == ST ? 0 : jp;
    // C's halo as the sequential reference sees it when it reaches this block
    const T* hc = P.inv[C] < P.inv[ib] ? h : hsnap;
    auto hv = [&](int x, int y) {
        const int c = memloc(x, y, C);
        return (x < 0 || x >= BW || y < 0 || y >= BW) ? hc[c] : h[c];
    };
    const int ii = memloc(cx, cy, C);
    const bool dry = !(h[ii] > eps && hv(cx - 1, cy) > eps && hv(cx + 1, cy) > eps && hv(cx, cy + 1) > eps &&
                       hv(cx, cy - 1) > eps);
    if (dry && !stage_off(loop_of(P, L, ib), corr)) {  // the stage flag is read alongside the cells
        const int w = edge_cell(s, -1, j, ib);
        h[w] = h[ii];
        zb[w] = zb[ii];
    }
}
template <class T>
__global__ __launch_bounds__(256) void k_amr_prolong(KParams P, T* h, T* zb, const T* hsnap, int level, DevLoop* L,
                                                     int corr) {
    amr_prolong<T>(P, h, zb, hsnap, level, L, corr, threadIdx.x, blockIdx.x);
}

// ----------------------------------------------------------------- fluxes
template <class T> struct StageIn {
    const T *h, *u, *v;
};
template <class T> struct FluxOut {
    T *Fhu, *Fqux, *Su, *Fqvx, *Fhv, *Fqvy, *Sv, *Fquy;
};

// The block and what surrounds it in LDS: h, zs, u, v at x, y in [-2, 17]
// (corners unused) and the slopes of the cells and of the halo ring; the
// faces take the slopes' place once they are formed (a third of the memory
// less, so four workgroups of the FP64 kernel share a CU instead of three),
// and the coarse blocks' cells that the linear prolongation needs stand there
// before the slopes are.  sh, sz: the h and zb of the coarser neighbours'
// cells that replace their halo cells in the source terms of the shared faces
// (src/Kurganov.cu:132-145).
constexpr int NPT = 33;  // prolongation points per side: see stage_point
template <class T> struct StageLds {
    Q4<T> q[20 * TP];
    union {
        struct {
            Q4<T> gx[16 * GXP];  // slopes along x of (h, zs, u, v)
            Q4<T> gy[18 * GYP];  // slopes along y of (h, zs, v, u)
        };
        struct {
            Q4<T> fx[BW * BW];   // X faces (Fhu, Fqux, Su, Fqvx)
            Q4<T> fy[BW * BW];   // Y faces (Fhv, Fqvy, Sv, Fquy)
        };
        T pt[4][4][NPT];         // h, u, v and the bed of the points
    };
    Q4<T> fe[2 * BW];  // the seventeenth X faces, then Y faces (before that: the EH_* cells of side s from 4 s)
    T sh[4][BW], sz[4][BW];
    T red[4];
};

// theta-minmod of src/Util_CPU.cu:243-263 by selection, for any theta.
template <class T> __device__ __forceinline__ T minmod2s(T theta, T s0, T s1, T s2) {
    const T d1 = theta * (s1 - s0), d2 = (s2 - s0) * T(0.5), d3 = theta * (s2 - s1);
    const bool up = s0 < s1 && s1 < s2, dn = s0 > s1 && s1 > s2;
    const T mn = dmin(dmin(d1, d2), d3), mx = dmax(dmax(d1, d2), d3);
    return up ? mn : dn ? mx : T(0.0);
}
// The slopes of a cell's four fields between its neighbours m and p.  FAST:
// the division by delta is a product with idelta, its hardware reciprocal.
template <bool FAST, class T>
__device__ __forceinline__ Q4<T> slopes4(T theta, const FixedDiv<T>& D, T idelta, const Q4<T>& m, const Q4<T>& c,
                                         const Q4<T>& p) {
    const Q4<T> g{minmod2s(theta, m.a, c.a, p.a), minmod2s(theta, m.b, c.b, p.b), minmod2s(theta, m.c, c.c, p.c),
                  minmod2s(theta, m.d, c.d, p.d)};
    return FAST ? Q4<T>{g.a * idelta, g.b * idelta, g.c * idelta, g.d * idelta} : div4(D, g);
}

// The h and zb of a coarser block's cell in the source term of a shared face;
// on: the face has one.
template <class T> struct SubVal {
    T h, z;
    bool on;
};

// One face between cell n (left or below) and cell i (src/Kurganov.cu:62-164,
// 1865-1911), from their (h, zs, un, ut) and slopes; Y faces come with u and v
// swapped.  FAST: hardware square roots and reciprocals for the IEEE ones.
// Returns whether the face is wet; lim receives its wave speed (0: none), or
// on spherical grids its CFL step.
template <class T, bool SPH, bool FAST>
__device__ __forceinline__ bool amr_face(T g, T CFL, T eps, T delta, T cm, T fm, const Q4<T>& qi, const Q4<T>& qn,
                                         const Q4<T>& gi, const Q4<T>& gn, const SubVal<T>& si, const SubVal<T>& sn,
                                         Q4<T>& F, T& lim) {
    using A = Ar<T, FAST>;
    const T epsi = epsi_of<T>();
    T hi = qi.a, hn = qn.a;
    const bool wet = hi > eps || hn > eps;
    const T dx = delta * T(0.5);
    T zi = qi.b - hi;
    const T zl = zi - dx * (gi.b - gi.a);
    T zn = qn.b - hn;
    const T zr = zn + dx * (gn.b - gn.a);
    const T zlr = smax(zl, zr);
    const T hl = hi - dx * gi.a;
    const T up = qi.c - dx * gi.c;
    const T hp = smax(T(0.0), hl + zl - zlr);
    const T hr = hn + dx * gn.a;
    const T um = qn.c + dx * gn.c;
    const T hm = smax(T(0.0), hr + zr - zlr);
    const T ga = g * T(0.5);
    const T cp = A::sqrt_(g * hp);
    const T cmo = A::sqrt_(g * hm);
    const T ap = smax(smax(up + cp, um + cmo), T(0.0));
    const T am = smin(smin(up - cp, um - cmo), T(0.0));
    const T ad = FAST ? A::rcp(ap - am) : plain_rcp(ap - am);
    const T qm = hm * um;
    const T qp = hp * up;
    const T hm2 = hm * hm;
    const T hp2 = hp * hp;
    const T a = smax(ap, -am);
    const T apm = ap * am;
    const bool flow = a > epsi;
    T fh = (ap * qm - am * qp + apm * (hp - hm)) * ad;
    T fu = (ap * (qm * um + ga * hm2) - am * (qp * up + ga * hp2) + apm * (qp - qm)) * ad;
    fh = flow ? fh : T(0.0);
    fu = flow ? fu : T(0.0);
    const T fv = (fh > T(0.0) ? qn.d + dx * gn.d : qi.d - dx * gi.d) * fh;
    if (SPH) {
        const T dlt = FAST ? delta * cm * A::rcp(fm) : delta * cm / fm;
        lim = !flow ? T(1.0) / epsi : FAST ? CFL * dlt * A::rcp(a) : CFL * dlt / a;
    } else {
        lim = flow && wet ? a : T(0.0);
    }
    if (si.on) {
        hi = si.h;
        zi = si.z;
    }
    if (sn.on) {
        hn = sn.h;
        zn = sn.z;
    }
    const T sl = ga * (hp * hp - hl * hl + (hl + hi) * (zi - zl));
    const T sr = ga * (hm * hm - hr * hr + (hr + hn) * (zn - zr));
    F.a = wet ? (SPH ? fm * fh : fh) : T(0.0);
    F.b = wet ? (SPH ? fm * (fu - sl) : fu - sl) : T(0.0);
    F.c = wet ? (SPH ? fm * (fu - sr) : fu - sr) : T(0.0);
    F.d = wet ? (SPH ? fm * fv : fv) : T(0.0);
    return wet;
}

// Metric terms of the faces of row y: cm of its X faces, cm and fm of the Y
// face below (y = 16: the top faces); 1 on Cartesian grids.
template <class T> struct FaceMetric {
    T cmx, cmy, fmy;
};
template <class T, bool SPH> __device__ __forceinline__ FaceMetric<T> face_metric(const KParams& P, int ib, int y) {
    FaceMetric<T> M{T(1.0), T(1.0), T(1.0)};
    if (SPH) {
        const T* m = (const T*)P.metric + (size_t)ib * METRIC_STRIDE;
        M.cmx = m[MET_CMX + (y < BW ? y : BW - 1)];
        M.cmy = m[MET_CMY + y];
        M.fmy = m[MET_FMY + y];
    }
    return M;
}

// Face position of side s at j: left and bottom faces are stored at the
// block's first cells, right and top faces at its halo.
__device__ __forceinline__ int face_at(int s, int j, int b) {
    return s == SL ? memloc(0, j, b) : s == SR ? memloc(BW, j, b) : s == SB ? memloc(j, 0, b) : memloc(j, BW, b);
}

// Face (s, j) of block ib after the fluxes: the restriction beside a finer
// neighbour and the boundary patch.
template <class T>
__device__ __forceinline__ void amr_fluxfix_side(const KParams& P, const FluxOut<T>& F, const StageIn<T>& E0,
                                                 const T* zb, const LoopState& L, int corr, int s, int j, int ib) {
    const int lev = P.level[ib];
    T* const A[4] = {s < 2 ? F.Fhu : F.Fhv, s < 2 ? F.Fqux : F.Fqvy, s < 2 ? F.Su : F.Sv, s < 2 ? F.Fqvx : F.Fquy};
    // coarse face = mean of the two fine faces (src/Halo.cu:1441-1529, 1766-1862)
    const Side S = side_of(P, s, ib);
    const int n = j < BW / 2 ? S.n1 : S.n2;
    if ((j < BW / 2 ? S.l1 : S.l2) > lev) {
        const int jj = (j & (BW / 2 - 1)) * 2;
        const int i = face_at(s, j, ib), il = face_at(s ^ 1, jj, n), itl = face_at(s ^ 1, jj + 1, n);
#pragma unroll
        for (int k = 0; k < 4; k++) A[k][i] = T(0.5) * (A[k][il] + A[k][itl]);
    }
    // wall boundary (noslipbndQ, src/Boundary.cu:1887-1891): no mass flux through
    // the boundary face and no normal-momentum flux difference in the edge cell
    if (S.n1 != ib && S.n2 != ib) return;
    const int ty = blk_btype(P, ib);
    if (ty == 0 || ty >= 2) {
        const int i = face_at(s, j, ib);
        if (ty >= 2) {
            // types 2 and 3 (bndFluxGPUSideCPU): the face's mass flux from the
            // step-start state (src/FlowCPU.cu:94, 187 pass evolv to both stages),
            // at totaltime + dt/2 (previous dt) or totaltime + dt, as the dt
            // reduction recorded them
            const int in = s == SL ? memloc(1, j, ib) : s == SR ? memloc(BW - 1, j, ib) : s == SB ? memloc(j, 1, ib)
                                                                                          : memloc(j, BW - 1, ib);
            const double ts = corr ? L.tcorr : L.tpred;
            const BSeg& G = P.seg[P.bseg[ib]];
            const int fx = s == SL ? 0 : s == SR ? BW : j, fy = s == SB ? 0 : s == ST ? BW : j;
            T q = A[0][i];
            if (bnd_flux<T>(P, s, ty, seg_level<T>(P, G, ts, ib, fx, fy), bnd_taper<T>(P, G, ts), zb[i] + E0.h[i],
                            E0.h[i], zb[in] + E0.h[in], E0.h[in], (s < 2 ? E0.u : E0.v)[in], q)) {
                A[0][i] = q;
                return;
            }
        }
        A[0][i] = T(0.0);
        if (s == SL) F.Su[memloc(1, j, ib)] = F.Fqux[i];
        else if (s == SR) F.Fqux[memloc(BW - 1, j, ib)] = F.Su[i];
        else if (s == SB) F.Sv[memloc(j, 1, ib)] = F.Fqvy[i];
        else F.Fqvy[memloc(j, BW - 1, ib)] = F.Sv[i];
    }
}

// --------------------------------------------------------------- advance
template <class T> struct AdvArgs {
    const T *h, *u, *v;        // stage state E of the tendencies
    const T *hold, *uold, *vold;  // state U^n the step starts from
    T *ho, *uo, *vo;           // output
    const T* zb;
    const T* cf;
};

// The tendencies of h, hu, hv of the blocks that do not wait for another
// block's faces, interior cells only (BSI values per block), between the
// predictor's stage and its advance.
template <class T> struct Tend {
    T *dh, *dhu, *dhv;
};

// A cell's values that the advance reads besides its tendencies.
template <class T> struct AdvIn {
    T hold, uold, vold, cf, zb;
};
template <class T> __device__ __forceinline__ AdvIn<T> adv_load(const AdvArgs<T>& A, int i, int corr) {
    AdvIn<T> X;
    X.hold = A.hold[i];
    X.uold = A.uold[i];
    X.vold = A.vold[i];
    X.cf = corr ? A.cf[i] : T(0);
    X.zb = corr ? A.zb[i] : T(0);
    return X;
}

// Tendencies of cell (x, y) of block ib (src/Advection.cu:160-254) from its
// stage state and its left, right, bottom and top faces; spherical grids take
// the row's metric terms.  The river discharges follow (AddRiverForcing after
// updateEV, src/FlowCPU.cu:120-124).
template <class T, bool SPH>
__device__ __forceinline__ void amr_tendencies(const KParams& P, T delta, T hi, T uui, T vvi, T Fhl, T Fhr, T Fhb,
                                               T Fht, T Fql, T Sr, T Fqb, T St, T Ftb, T Ftt, T Ftl, T Ftr,
                                               double tstart, int ib, int x, int y, T& dh, T& dhu, T& dhv) {
    const T* met = (const T*)P.metric + (size_t)ib * METRIC_STRIDE;
    const T fc = SPH ? met[MET_FC + y] : T(P.fc);
    const T cm = SPH ? met[MET_CME + y] : T(1.0);
    const T cmdinv = T(1.0) / (cm * delta);
    dh = river_inflow<T>(P, ib, x, y, tstart, T(-1.0) * (Fhr - Fhl + Fht - Fhb) * cmdinv);
    dhu = (Fql + Ftb - Sr - Ftt) * cmdinv + fc * hi * vvi;
    dhv = (Fqb + Ftl - St - Ftr) * cmdinv - fc * hi * uui;
    if (SPH) {  // the metric differences, zero on Cartesian grids
        const T fmu = T(1.0), fmup = T(1.0);
        const T fmv = met[MET_FMV + y], fmvp = met[MET_FMVP + y];
        const T ga = T(0.5) * T(P.g);
        const T dmdl = (fmup - fmu) / (cm * delta);
        const T dmdt = (fmvp - fmv) / (cm * delta);
        const T fG = vvi * dmdl - uui * dmdt;
        dhu += hi * (ga * hi * dmdl + fG * vvi);
        dhv += hi * (ga * hi * dmdt - fG * uui);
    }
}

// The update of a cell by its tendencies (src/Advection.cu:332-385; the drying
// limiter in double), and in the corrector the bottom friction
// (src/Friction.cu:89-148), cleanup and the implicit rain
// (src/Updateforcing.cu:530-581).
template <class T>
__device__ __forceinline__ void amr_update(const KParams& P, const AdvArgs<T>& A, const AdvIn<T>& X, T dhi, T dhu,
                                           T dhv, const LoopState& L, int corr, int i, int ib, int x, int y) {
    const T dt = corr ? T(L.dt) : T(L.dt) * T(0.5);
    const T g = T(P.g);
    const T eps = T(P.eps);
    const T hold = X.hold;
    const T edt = P.ForceMassConserve ? dt : dry_step(dt, hold, dhi, eps, P.eps);
    T ho = hold + edt * dhi, uo, vo;
    if (ho > eps) {
        uo = (hold * X.uold + edt * dhu) / ho;
        vo = (hold * X.vold + edt * dhv) / ho;
    } else {
        uo = T(0.0);
        vo = T(0.0);
    }
    if (corr) {
        // bottom friction, src/Friction.cu:89-148
        if (ho > eps) {
            const T normu = sqrt(uo * uo + vo * vo);
            const T cfv = X.cf;
            T cfi = T(0);
            if (P.frictionmodel == 0) {
                cfi = cfv;
            } else if (P.frictionmodel == 1) {
                const T ee = T(2.71828182845905);
                const T Hbar = ho / cfv;
                if (Hbar <= ee) cfi = T(1.0) / (T(0.46) * Hbar);
                else cfi = T(1.0) / (T(2.5) * (log(Hbar) - T(1.0) + T(1.359) / Hbar));
                cfi = cfi * cfi;
            } else if (P.frictionmodel == -1) {
                cfi = g * cfv * cfv / cbrt(ho);
            }
            const T tb = cfi * normu / ho * dt;
            uo = uo / (T(1.0) + tb);
            vo = vo / (T(1.0) + tb);
        }
        // cleanup then implicit uniform rain, src/Updateforcing.cu:530-581
        if (P.rain_on) {
            const T act = (double)X.zb < P.mask ? T(1.0) : T(0.0);
            T rainhh = rain_depth<T>(P, L, ib, x, y, T(L.dt)) * act;
            const T qvol = ho / (ho + rainhh);
            const bool wet = (double)ho > P.eps;
            ho = ho + rainhh;
            if (wet) {
                uo = uo * qvol;
                vo = vo * qvol;
            }
        }
    }
    A.ho[i] = ho;
    A.uo[i] = uo;
    A.vo[i] = vo;
    if (corr && P.hmax) {  // running maximum depth (batch members)
        const float hv = (float)ho;
        if (hv > P.hmax[i]) P.hmax[i] = hv;
    }
}

// Whether block ib's stage ends in the deferred fix-up (its faces stored,
// restricted beside finer blocks and patched on open boundaries, then its
// advance) instead of in the stage's own launch: it has a finer neighbour, or
// a boundary side in a run with open segments, whose faces follow the dt
// reduction.  info: any of the block's level words (REC_* flags).  The host's
// list of these blocks (P.fix) follows the same rule.
__device__ __forceinline__ bool fix_block(const KParams& P, int info) {
    return P.fix_all || (info & REC_FINER) || (P.bopen && (info & REC_EDGE));
}

// One wave per block, thread (side, j): the block's halo for the stage, on
// meshes of four levels and more, whose wet/dry prolongation runs level by
// level (k_amr_prolong).  A block writes its own halo only and reads other
// blocks' interior cells and the bed halo cells that the prolongation leaves
// alone (beside a finer block).
template <class T>
__global__ __launch_bounds__(64) void k_amr_halo_refine(KParams P, T* h, T* u, T* v, T* zb, T* hsnap, DevLoop* L,
                                                        int corr) {
    const int ib = P.active[blockIdx.x];
    const DevLoop* Lm = loop_of(P, L, ib);
    const int s = threadIdx.x >> 4, j = threadIdx.x & 15;
    const HaloVals<T> o = amr_halo_refine<T>(P, h, u, v, zb, hsnap != nullptr, s, j, ib, P.level[ib]);
    if (stage_off(Lm, corr)) return;  // the values are formed before the flag is known
    const int w = edge_cell(s, -1, j, ib);
    h[w] = o.h;
    u[w] = o.u;
    v[w] = o.v;
    if (hsnap) hsnap[w] = o.hs;
    if (o.zbset) zb[w] = o.zb;
}

// Tile position of depth d (-1 the halo, -2 beyond it) of side s at j.
__device__ __forceinline__ int side_tix(int s, int d, int j) {
    return s == SL ? tix(d, j) : s == SR ? tix(BW - 1 - d, j) : s == SB ? tix(j, d) : tix(j, BW - 1 - d);
}

// The coarse cells that the linear prolongation of side s (beside the coarser
// block C) reads, one per lane k: a half side of C is eight edge cells, and
// their neighbours make 26 points --
//   0..9    C's edge cells from one before the half to one after it (an end
//           beyond C's side is C's halo on the adjoining side),
//   10..17  the cells behind them,
//   18..25  C's halo in front of them;
// 26..30 the five points (a cell of D and its four neighbours) behind C's
//         halo at the end of its side, where the block D there is coarser than
//         C,
//   31    C's halo at that end, behind point 0 or 9,
//   32    C's cell behind the edge cell at the other end of the half.
// 26..31 give C's halo at the end of the half as C's own halo stage leaves it
// (k_amr_stage), which the sequential reference's wet/dry prolongation tests
// and the cells beyond the halo are interpolated from.
// side_end gives that halo: side p of C, position je beside the shared side.
struct SideEnd {
    int p, je;
    Side E;  // side p of C
};
__device__ __forceinline__ void side_end(int s, bool lo, int& p, int& je) {
    p = s < 2 ? (lo ? SB : ST) : (lo ? SL : SR);
    je = (s == SL || s == SB) ? BW - 1 : 0;
}
__device__ __forceinline__ SideEnd side_end(const KParams& P, int s, const Side& S) {
    SideEnd e;
    side_end(s, S.back, e.p, e.je);
    e.E = side_of(P, e.p, S.n1);
    return e;
}
// Cell of C at depth d from its side facing side s of the block, at position a.
__device__ __forceinline__ void facing_cell(int s, int d, int a, int& x, int& y) {
    const int n = (s == SL || s == SB) ? BW - 1 - d : d;
    x = s < 2 ? n : a;
    y = s < 2 ? a : n;
}
template <class T>
__device__ __forceinline__ HaloPt<T> stage_point(const KParams& P, int s, int k, const Side& S) {
    const int j0 = S.back ? 0 : BW / 2;
    int x, y, b = S.n1, lev = S.l1;
    if (k < 26 || k > 30) {
        const int d = k < 10 ? 0 : k < 18 || k > 30 ? 1 : -1;
        const int a = k < 10   ? j0 - 1 + k
                      : k < 18 ? j0 + k - 10
                      : k < 26 ? j0 + k - 18
                      : k < 32 ? (S.back ? -1 : BW)
                               : (S.back ? BW / 2 : BW / 2 - 1);
        facing_cell(s, d, a, x, y);
    } else {
        const SideEnd e = side_end(P, s, S);
        const Side& E = e.E;
        if (!(E.l1 < S.l1)) {  // no coarser block there: any cell of C
            facing_cell(s, 0, j0, x, y);
        } else {
            const int a = e.je / 2 + (E.back ? 0 : BW / 2);
            facing_cell(e.p, 0, a, x, y);
            const int m = k - 26;
            x += m == 1 ? -1 : m == 2 ? 1 : 0;
            y += m == 3 ? -1 : m == 4 ? 1 : 0;
            b = E.n1;
            lev = E.l1;
        }
    }
    return pt_recipe<T>(P, x, y, b, lev);
}

// The recipes of the sides that are not beside blocks of the block's own
// level: NPT entries a side, of a coarse side its points, of another the halo
// cells (0..15) and the cells beyond them (16..31).  They depend on the mesh
// only and are formed once for it: to form them in every stage again took a
// chain of dependent loads through the neighbours' records and half of the
// stage's 44 to 53 KB of code, more for the two stages than the instruction
// cache holds (1,607 blocks in FP32: 23 us a stage, now 17; the same blocks
// taken as all of one level, wrongly, 13).  An entry is four cells (P.rcell) and a code with
// the cell of the bed (P.rmeta).
enum {
    RC_KIND = 3, RC_SET = 2, RC_WD = 1 << 5, RC_SIDE = 6,  // G_* kind; w3 set; wet/dry restriction; its side
    RC_FIRST = 1 << 8,                                     // coarse sides: C comes before the block in the active list
    RC_END = 16                                            // and the level of the block at the end of the half
};
static_assert(4 * NPT == RECIPES, "");
__global__ __launch_bounds__(192) void k_amr_recipes(KParams P, int4* rcell, int2* rmeta) {
    const int t = threadIdx.x, ib = P.active[blockIdx.x], s = t / NPT, k = t % NPT;
    if (s > 3) return;
    const int lev = P.level[ib];
    const Side S = side_of(P, s, ib);
    const bool coarse = S.l1 < lev;
    if (!coarse && k >= 32) return;
    HaloPt<float> r;
    int code = 0;
    if (coarse) {
        r = stage_point<float>(P, s, k, S);
        const SideEnd e = side_end(P, s, S);
        code = (P.inv[S.n1] < P.inv[ib] ? RC_FIRST : 0) | (e.E.l1 & 0xff) << RC_END;
    } else if (k < 16) {
        r.g = fill_recipe<float>(P, S, s, k, ib, lev);
        r.wd = wetdry_recipe(P, S, s, k, ib, lev);
    } else {
        r.g = far_recipe<float>(S, s, k - 16, ib, lev);
        r.wd.on = 0;
        r.wd.w = r.g.i[0];
    }
    // the side whose patch a restriction reads: the mean's cells are that patch's, in its side's order
    int rs = s;
    if (coarse) {
        const int x = r.wd.w % BS % MW, y = r.wd.w % BS / MW;
        rs = x == 0 ? SL : x == MW - 1 ? SR : y == 0 ? SB : ST;
    }
    const size_t e = ((size_t)ib * 4 + s) * NPT + k;
    rcell[e] = make_int4(r.g.i[0], r.g.i[1], r.g.i[2], r.g.i[3]);
    rmeta[e] = make_int2(code | r.g.kind | r.g.set << RC_SET | (r.wd.on ? RC_WD : 0) | rs << RC_SIDE, r.wd.w);
}

// What a wave keeps of C's halo at the end of its half side: the cell beside the
// shared side as this block's prolongation sees it, as C's own stage leaves it,
// and the cell behind that.
enum { EH_SEEN = 0, EH_FACING = 1, EH_BEHIND = 2, EH_N = 3 };

// Orders a wave's LDS writes before its lanes' reads of one another's.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// A stage of a block in one workgroup: halo, slopes, faces, tendencies, and in
// the corrector the advance.
//
// Wave s gathers side s: its halo cells (lanes 0-15) and the cells beyond the
// halo that the limited slope at the halo reads (src/Gradients.cu:2713-3294,
// lanes 32-47), by the mesh's recipes where the neighbours are of another
// level; the side's kind is uniform over its wave.  Beside a coarser block it
// gathers the points of stage_point (lanes 0-32) and forms from them the linear
// reconstruction and the wet/dry prolongation (src/Halo.cu:1044-1405,
// src/ConserveElevation.cu:80-205,451-482), the cells beyond and the source
// substitutions (lanes 48-63).  HALO: the halo is formed here; otherwise it
// stands in the Model arrays (four levels and more).  The slopes, faces and
// tendencies are those of the one-level tile.
//
// A block that needs no other block's faces has its tendencies stored (the
// predictor, whose dt is not known yet) or is advanced here (the corrector:
// it writes the state's interior cells, which no other block of the corrector
// stage reads); beside a coarser block it leaves the shared faces in the face
// arrays.  The others (fix_block) store all their faces for the fix-up.
// Everything global is read before the stage flag is tested.
template <class T, bool SPH, bool FAST, bool HALO, int corr>
__global__ __launch_bounds__(256, sizeof(T) == 8 ? 4 : 7) void k_amr_stage(KParams P, AdvArgs<T> A, T* zb,
                                                                           FluxOut<T> F, Tend<T> D, DevLoop* L) {
    __shared__ StageLds<T> S;
    const int t = threadIdx.x, x = t & 15, y = t >> 4;
    const int ib = ldu(P.active, xcd_range(blockIdx.x % NXCD, P.nblk).start + blockIdx.x / NXCD);
    DevLoop* Lm = loop_of(P, L, ib);
    const int lev = ldu(P.level, ib);
    int nb[8], info[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
        nb[k] = ldu(P.nbr, ib * NBR + k);
        info[k] = ldu(P.nbr, ib * NBR + 8 + k);
    }
    bool cs[4];  // the side is beside a coarser block
#pragma unroll
    for (int k = 0; k < 4; k++) cs[k] = rec_level(info[2 * k]) < lev;
    const bool fix = fix_block(P, info[0]);
    const bool prolong = P.wetdryfix && P.maxlevel > P.minlevel;
    const T theta = T(P.theta), eps = T(P.eps);
    const T delta = calcres(T(P.delta0), lev);
    const T idelta = Ar<T, FAST>::rcp(delta);
    const FixedDiv<T> by_delta = fixed_div(delta);

    // the block's own cell
    const int c = memloc(x, y, ib);
    const T h0 = A.h[c], z0 = zb[c], u0 = A.u[c], v0 = A.v[c];
    AdvIn<T> X;
    if (corr && !fix) X = adv_load(A, c, 1);

    // the wave's side
    const int s = __builtin_amdgcn_readfirstlane(t >> 6), l = t & 63, j = l & 15;
    const Side sd = side_of_uniform(P, s, ib);
    const bool coarse = sd.l1 < lev;
    const bool is_far = (l >> 4) == 2, is_sub = (l >> 4) == 3;
    const int w = edge_cell(s, -1, j, ib);
    Q4<T> r;  // the value of the lane's point: h, zs, u, v (halo cells: zs without the bed yet)
    T zw = T(0), zown = T(0);  // the bed of the lane's point, and of the block's own halo cell
    int ends = 0;              // the coarse side's code
    r.a = r.b = r.c = r.d = T(0);
    const bool same = (sd.n1 == ib && sd.n2 == ib) || (sd.n1 != ib && sd.l1 == lev && sd.l2 == lev);
    if (l < 16) zown = zw = zb[w];
    if (same) {
        if (l < 16 || is_far) {
            const int i = sd.n1 == ib ? edge_cell(s, 0, j, ib) : edge_cell(s ^ 1, is_far ? 1 : 0, j, sd.n1);
            r.a = A.h[i];
            r.b = zb[i];
            r.c = A.u[i];
            r.d = A.v[i];
            r.b = r.b + r.a;
        }
        if (!HALO && l < 16) {
            r.a = A.h[w];
            r.c = A.u[w];
            r.d = A.v[w];
        }
    } else if (HALO) {
        const int e = (ib * 4 + s) * NPT;
        if (coarse) ends = ldu((const int*)P.rmeta, 2 * e);
        if (coarse ? l < NPT : l < 16 || is_far) {
            const int k = e + (coarse || l < 16 ? l : l - 16);
            const int4 n = P.rcell[k];
            const int2 m = P.rmeta[k];
            const int kind = m.x & RC_KIND;
            T H[4], Z[4], U[4], V[4];
            auto load = [&](int q, int c) {
                H[q] = A.h[c];
                Z[q] = zb[c];
                U[q] = A.u[c];
                V[q] = A.v[c];
            };
            load(0, n.x);
            if (coarse) zw = zb[m.y];
            if (kind != G_COPY) {
                load(1, n.y);
                load(2, n.z);
                load(3, n.w);
            }
            r = Q4<T>{H[0], Z[0] + H[0], U[0], V[0]};
            if (kind == G_MEAN4) {
                auto mean = [](const T* z) { return T(0.25) * (z[0] + z[1] + z[2] + z[3]); };
                r.a = mean(H);
                r.c = mean(U);
                r.d = mean(V);
                if (is_far) {
#pragma unroll
                    for (int q = 0; q < 4; q++) Z[q] = Z[q] + H[q];
                    r.b = mean(Z);
                }
                if ((m.x & RC_WD) && P.wetdryfix) {
                    // the patch's cells in the restriction's order (lower left, right, top, top right)
                    const int rs = (m.x >> RC_SIDE) & 3;
                    const bool lo = rs == SL || rs == SB, xs = rs < 2;
                    auto patch = [&](const T* z, T* o) {
                        o[0] = lo ? z[1] : z[0];
                        o[1] = xs ? (lo ? z[0] : z[1]) : (lo ? z[3] : z[2]);
                        o[2] = xs ? (lo ? z[3] : z[2]) : (lo ? z[0] : z[1]);
                        o[3] = lo ? z[2] : z[3];
                    };
                    T hh[4], zz[4];
                    patch(H, hh);
                    patch(Z, zz);
                    r.a = wetdry_apply(eps, hh, zz, zw, r.a);
                }
            } else if (kind == G_W3) {
                T a, b, c;
                w3_weights((m.x >> RC_SET) & 7, a, b, c);
                auto w3 = [&](const T* z) { return a * z[0] + b * z[1] + c * z[2]; };
                r.a = w3(H);
                r.c = w3(U);
                r.d = w3(V);
            }
        }
    } else {
        Gather<T> g;
        if (is_far) {
            g = far_recipe<T>(sd, s, j, ib, lev);
        } else if (is_sub) {
            // the coarse cell next to the face (where the side is coarse; read anyway)
            int cx, cy;
            facing_cell(s, 0, coarse ? j / 2 + (sd.back ? 0 : BW / 2) : 0, cx, cy);
            g = g_copy<T>(memloc(cx, cy, sd.n1));
        } else {
            g = g_copy<T>(w);
        }
        T H[4], Z[4], U[4], V[4];
        g_load(g, A.h, H);
        g_load(g, zb, Z);
        g_load(g, A.u, U);
        g_load(g, A.v, V);
        r.a = g_apply(g, H);
        r.c = g_apply(g, U);
        r.d = g_apply(g, V);
        if (is_far) {
#pragma unroll
            for (int m = 0; m < 4; m++) Z[m] = Z[m] + H[m];
            r.b = g_apply(g, Z);
        } else {
            r.b = Z[0];
        }
    }
    if (stage_off(Lm, corr)) return;  // the workgroup's one block: all threads leave together

    const Q4<T> q{h0, z0 + h0, u0, v0};
    S.q[tix(x, y)] = q;
    if (HALO && coarse) {
        // the side's own wave passes its points through LDS: in order within a wave, no barrier
        if (l < NPT) {
            S.pt[s][0][l] = r.a;
            S.pt[s][1][l] = r.c;
            S.pt[s][2][l] = r.d;
            S.pt[s][3][l] = zw;
        }
        wave_sync();
        // the linear reconstructions: lanes 0-15 of the halo cells, lanes 48-50 of C's halo at the end of
        // the half (the EH_* cells, to S.fe[4 s + EH_*])
        int p = s, jr = j;
        const int m = j / 2, lend = (int)(signed char)(ends >> RC_END);
        const bool lo = s == SL || s == SB;  // the side faces the neighbour's high end
        const int kend = l == 48 + EH_BEHIND ? 31 : sd.back ? 0 : 9;
        Q4<T> o{T(0), T(0), T(0), T(0)};
        T f0[5];
        if (l < 16 || (is_sub && j < EH_N)) {
            int k[5], lv = lev, lc = sd.l1;
            if (l < 16) {
                // the points of the coarse cell m of the half and of its neighbours in x and y
                const int in = 10 + m, out = 18 + m, before = m, after = m + 2;
                k[0] = m + 1;
                k[1] = s < 2 ? (lo ? in : out) : before;
                k[2] = s < 2 ? (lo ? out : in) : after;
                k[3] = s < 2 ? before : (lo ? in : out);
                k[4] = s < 2 ? after : (lo ? out : in);
            } else {
#pragma unroll
                for (int n = 0; n < 5; n++) k[n] = 26 + n;
                side_end(s, sd.back, p, jr);
                if (j == EH_BEHIND) jr += jr == 0 ? 1 : -1;
                lv = sd.l1;
                lc = lend;
            }
            T f[2][5];
#pragma unroll
            for (int n = 0; n < 5; n++) {
                f0[n] = S.pt[s][0][k[n]];
                f[0][n] = S.pt[s][1][k[n]];
                f[1][n] = S.pt[s][2][k[n]];
            }
            o.a = refine_from(P, p, jr, lv, lc, f0);
            o.c = refine_from(P, p, jr, lv, lc, f[0]);
            o.d = refine_from(P, p, jr, lv, lc, f[1]);
        }
        auto dry = [&]() { return !(f0[0] > eps && f0[1] > eps && f0[2] > eps && f0[4] > eps && f0[3] > eps); };
        if (is_sub) {
            S.sh[s][j] = S.pt[s][0][m + 1];
            S.sz[s][j] = S.pt[s][3][m + 1];
            if (j < EH_N) {
                // Beside a coarser block D it is the linear reconstruction, or, where the wet/dry
                // prolongation applies, D's cell (both depths lie over one cell of D); C's own workgroup
                // may be writing the bed of that halo cell, but only where it becomes the bed of D's cell,
                // which is taken from D here.
                if (!(lend < sd.l1)) o = Q4<T>{S.pt[s][0][kend], T(0), S.pt[s][1][kend], S.pt[s][2][kend]};
                o.b = S.pt[s][3][kend];
                if (lend < sd.l1 && prolong && (j != EH_SEEN || (ends & RC_FIRST)) && dry()) {
                    o.a = f0[0];
                    o.b = S.pt[s][3][26];
                }
                o.b = o.b + o.a;
                S.fe[4 * s + j] = o;
            }
        }
        wave_sync();
        if (l < 16) {
            T zo = zown;
            if (prolong) {
                // C's halo at the end, prolonged if C comes before this block in the active list
                if (m == (sd.back ? 0 : BW / 2 - 1)) {
                    const T ha = S.fe[4 * s + EH_SEEN].a;
                    if (s < 2) (sd.back ? f0[3] : f0[4]) = ha;
                    else (sd.back ? f0[1] : f0[2]) = ha;
                }
                if (dry()) {
                    o.a = f0[0];
                    zo = S.pt[s][3][m + 1];
                    zb[w] = zo;
                }
            }
            o.b = zo + o.a;
            S.q[side_tix(s, -1, j)] = o;
        } else if (is_far) {
            // the cells beyond the halo: bilinear from C's cells at depths 0 and 1 (far_recipe), at the
            // end of the half C's halo
            const int cj = (j + 1) / 2;
            const T b = cj * 2 > j ? T(0.25) : T(0.75);
            auto at = [&](int k) {
                const T h = S.pt[s][0][k];
                return Q4<T>{h, S.pt[s][3][k] + h, S.pt[s][1][k], S.pt[s][2][k]};
            };
            Q4<T> p0 = at(cj + 1), q0 = at(cj), p1 = at(cj < BW / 2 ? 10 + cj : sd.back ? 32 : 31),
                  q1 = at(cj > 0 ? 9 + cj : sd.back ? 31 : 32);
            if (sd.back && cj == 0) {
                q0 = S.fe[4 * s + EH_FACING];
                q1 = S.fe[4 * s + EH_BEHIND];
            }
            if (!sd.back && cj == BW / 2) {
                p0 = S.fe[4 * s + EH_FACING];
                p1 = S.fe[4 * s + EH_BEHIND];
            }
            // bilinear(q11, q12, q21, q22, x, y) with the side's corner order
            const Q4<T> c12 = s < 2 ? (lo ? p1 : p0) : (lo ? q0 : q1), c21 = s < 2 ? (lo ? q0 : q1) : (lo ? p1 : p0);
            const Q4<T> c11 = lo ? q1 : q0, c22 = lo ? p0 : p1;
            const T a = lo ? T(0.75) : T(0.25), bx = s < 2 ? a : b, by = s < 2 ? b : a;
            S.q[side_tix(s, -2, j)] = Q4<T>{bilinear(c11.a, c12.a, c21.a, c22.a, bx, by),
                                            bilinear(c11.b, c12.b, c21.b, c22.b, bx, by),
                                            bilinear(c11.c, c12.c, c21.c, c22.c, bx, by),
                                            bilinear(c11.d, c12.d, c21.d, c22.d, bx, by)};
        }
    } else {
        if (is_far) S.q[side_tix(s, -2, j)] = r;
        if (is_sub && coarse) {
            S.sh[s][j] = r.a;
            S.sz[s][j] = r.b;
        }
        if (l < 16) {
            r.b = zw + r.a;
            S.q[side_tix(s, -1, j)] = r;
            // open boundaries take the step-start depth of the halo (amr_fluxfix_side: the right and top faces)
            if (HALO && !corr && P.bopen && (sd.n1 == ib || sd.n2 == ib)) const_cast<T*>(A.h)[w] = r.a;
        }
    }
    __syncthreads();

    // slopes: the thread's own cell, and the halo ring on wave 2 (lanes 0-31 along x, 32-63 along y)
    const Q4<T> gxo = slopes4<FAST>(theta, by_delta, idelta, S.q[tix(x - 1, y)], q, S.q[tix(x + 1, y)]);
    S.gx[gxi(x, y)] = gxo;
    Q4<T> gyo = slopes4<FAST>(theta, by_delta, idelta, S.q[tix(x, y - 1)], q, S.q[tix(x, y + 1)]);
    {
        const T a = gyo.c;  // stored as (h, zs, v, u)
        gyo.c = gyo.d;
        gyo.d = a;
        S.gy[gyi(x, y)] = gyo;
    }
    if (s == 2) {
        const bool isx = l < 32;
        const int o = (l & 16) ? BW : -1;
        const int ci = isx ? tix(o, j) : tix(j, o), d = isx ? 1 : TP;
        const Q4<T> g = slopes4<FAST>(theta, by_delta, idelta, S.q[ci - d], S.q[ci], S.q[ci + d]);
        if (isx) S.gx[gxi(o, j)] = g;
        else S.gy[gyi(j, o)] = Q4<T>{g.a, g.b, g.d, g.c};
    }
    __syncthreads();

    // faces: the cell's left and bottom ones, and the seventeenth ones on wave 3 (lanes 0-15 X, 16-31 Y)
    const T g = T(P.g), CFL = T(P.CFL), inv_epsi = T(1.0) / epsi_of<T>(), epsw = eps + epsi_of<T>();
    const SubVal<T> none{T(0), T(0), false};
    auto sub = [&](int k, int jj, bool here) {
        return here && cs[k] ? SubVal<T>{S.sh[k][jj], S.sz[k][jj], true} : none;
    };
    auto swap_uv = [](const Q4<T>& a) { return Q4<T>{a.a, a.b, a.d, a.c}; };
    const FaceMetric<T> M = face_metric<T, SPH>(P, ib, y);
    Q4<T> Fl, Fb;
    T lx, ly;
    const bool wx = amr_face<T, SPH, FAST>(g, CFL, epsw, delta, M.cmx, T(1.0), q, S.q[tix(x - 1, y)], gxo,
                                           S.gx[gxi(x - 1, y)], none, sub(SL, y, x == 0), Fl, lx);
    finish(Fl);
    const bool wy = amr_face<T, SPH, FAST>(g, CFL, epsw, delta, M.cmy, M.fmy, swap_uv(q), swap_uv(S.q[tix(x, y - 1)]),
                                           gyo, S.gy[gyi(x, y - 1)], none, sub(SB, x, y == 0), Fb, ly);
    finish(Fb);
    const bool edge = s == 3 && l < 32, ex = l < 16;
    if (edge) {
        const FaceMetric<T> Me = face_metric<T, SPH>(P, ib, ex ? j : BW);
        const int ci = ex ? tix(BW, j) : tix(j, BW);
        Q4<T> qi = S.q[ci], qn = S.q[ci - (ex ? 1 : TP)];
        if (!ex) {
            qi = swap_uv(qi);
            qn = swap_uv(qn);
        }
        const Q4<T> gi = ex ? S.gx[gxi(BW, j)] : S.gy[gyi(j, BW)], gn = ex ? S.gx[gxi(BW - 1, j)] : S.gy[gyi(j, BW - 1)];
        SubVal<T> se = none;
        if (ex ? cs[SR] : cs[ST]) se = SubVal<T>{S.sh[ex ? SR : ST][j], S.sz[ex ? SR : ST][j], true};
        T le;
        Q4<T> Fe;
        (void)amr_face<T, SPH, FAST>(g, CFL, epsw, delta, ex ? Me.cmx : Me.cmy, ex ? T(1.0) : Me.fmy, qi, qn, gi, gn, se,
                                     none, Fe, le);
        S.fe[l] = Fe;
    }
    __syncthreads();  // the slopes are read: the faces take their place
    S.fx[t] = Fl;
    S.fy[t] = Fb;
    if (!corr) {
        // dtmax of the cell: its X face, then its Y face, a dry face resetting it to 1/epsi
        // (src/Kurganov.cu:1488-1491); off the sphere every face has the same cell size, so the block's
        // largest wave speed gives its smallest step (the rounded division is monotone)
        T d;
        if (SPH) {
            d = wx ? (lx < tmax_of<T>() ? lx : tmax_of<T>()) : inv_epsi;
            d = wy ? (ly < d ? ly : d) : inv_epsi;
        } else {
            d = wy ? -smax(lx, ly) : T(0.0);
        }
        T m = block_min(d, S.red, t);
        if (!SPH) {
            m = -m > T(0.0) ? (FAST ? CFL * delta * Ar<T, FAST>::rcp(-m) : CFL * delta / -m) : inv_epsi;
            m = m < inv_epsi ? m : inv_epsi;
        }
        if (t == 0) slot_min(Lm, blockIdx.x, m);
    } else {
        __syncthreads();
    }

    // faces that other launches read: all of a fix-up block's, else those beside a coarser block
    auto put = [&](const Q4<T>& f, bool xface, int i) {
        (xface ? F.Fhu : F.Fhv)[i] = f.a;
        (xface ? F.Fqux : F.Fqvy)[i] = f.b;
        (xface ? F.Su : F.Sv)[i] = f.c;
        (xface ? F.Fqvx : F.Fquy)[i] = f.d;
    };
    if (fix || (cs[SL] && x == 0)) put(Fl, true, c);
    if (fix || (cs[SB] && y == 0)) put(Fb, false, c);
    if (edge && (fix || (ex ? cs[SR] : cs[ST]))) put(S.fe[l], ex, ex ? memloc(BW, j, ib) : memloc(j, BW, ib));
    if (fix) return;

    const Q4<T> Fr = x < BW - 1 ? S.fx[t + 1] : S.fe[y], Ft = y < BW - 1 ? S.fy[t + BW] : S.fe[BW + x];
    T Fhl = Fl.a, Fhr = Fr.a, Fql = Fl.b, Sr = Fr.c;
    T Fhb = Fb.a, Fht = Ft.a, Fqb = Fb.b, St = Ft.c;
    if ((info[0] & REC_EDGE) && blk_btype(P, ib) == 0) {
        // walls (noslipbndQ, src/Boundary.cu:1887-1891): no mass flux through the boundary face and no
        // normal-momentum flux difference in the edge cell
        if (x == 0 && (nb[0] == ib || nb[1] == ib)) { Fhl = T(0.0); Sr = Fql; }
        if (x == BW - 1 && (nb[2] == ib || nb[3] == ib)) { Fhr = T(0.0); Fql = Sr; }
        if (y == 0 && (nb[4] == ib || nb[5] == ib)) { Fhb = T(0.0); St = Fqb; }
        if (y == BW - 1 && (nb[6] == ib || nb[7] == ib)) { Fht = T(0.0); Fqb = St; }
    }
    T dh, dhu, dhv;
    amr_tendencies<T, SPH>(P, delta, h0, u0, v0, Fhl, Fhr, Fhb, Fht, Fql, Sr, Fqb, St, Fb.d, Ft.d, Fl.d, Fr.d,
                           corr ? Lm->tstart : Lm->totaltime, ib, x, y, dh, dhu, dhv);
    if (corr) {
        amr_update<T>(P, A, X, dh, dhu, dhv, *Lm, 1, c, ib, x, y);
    } else {
        const int k = ib * BSI + t;
        D.dh[k] = dh;
        D.dhu[k] = dhu;
        D.dhv[k] = dhv;
    }
}

// The fix-up of a block's stored faces (beside finer blocks: the finer
// neighbours' faces, which no launch of this kernel writes; on the domain
// edge), then its advance.
template <class T, bool SPH>
__device__ __forceinline__ void fix_advance(const KParams& P, const StageIn<T>& E0, const AdvArgs<T>& A,
                                            const FluxOut<T>& F, const LoopState& L, int corr, int t, int ib) {
    const int x = t & 15, y = t >> 4;
    const int i = memloc(x, y, ib), ir = memloc(x + 1, y, ib), it = memloc(x, y + 1, ib);
    const AdvIn<T> X = adv_load(A, i, corr);
    const T h = A.h[i], u = A.u[i], v = A.v[i];
    if (!L.go) return;  // the workgroup's one block: all threads leave together
    if (t < 64) amr_fluxfix_side<T>(P, F, E0, A.zb, L, corr, t >> 4, t & 15, ib);
    __syncthreads();
    T dh, dhu, dhv;
    amr_tendencies<T, SPH>(P, calcres(T(P.delta0), P.level[ib]), h, u, v, F.Fhu[i], F.Fhu[ir], F.Fhv[i], F.Fhv[it],
                           F.Fqux[i], F.Su[ir], F.Fqvy[i], F.Sv[it], F.Fquy[i], F.Fquy[it], F.Fqvx[i], F.Fqvx[ir],
                           L.tstart, ib, x, y, dh, dhu, dhv);
    amr_update<T>(P, A, X, dh, dhu, dhv, L, corr, i, ib, x, y);
}

// The predictor's advance: U* = U + dt/2 L(U) from the stored tendencies, or
// from the fixed-up faces, with the step's dt.  REDUCED: the reduction was a
// launch before (a block of a batch finds its member's state in L); otherwise
// every workgroup works it out from the slots (step_state).
template <class T, bool SPH, bool REDUCED>
__global__ __launch_bounds__(256) void k_amr_advance(KParams P, StageIn<T> E0, AdvArgs<T> A, FluxOut<T> F, Tend<T> D,
                                                     DevLoop* L, DevLoop* Lnext, int mode) {
    const int ib = ldu(P.active, xcd_range(blockIdx.x % NXCD, P.nblk).start + blockIdx.x / NXCD);
    const int t = threadIdx.x;
    const int i = memloc(t & 15, t >> 4, ib), k = ib * BSI + t;
    const bool fix = fix_block(P, ldu(P.nbr, ib * NBR + 8));
    AdvIn<T> X;
    T dh = T(0), dhu = T(0), dhv = T(0);
    if (!fix) {
        X = adv_load(A, i, 0);
        dh = D.dh[k];
        dhu = D.dhu[k];
        dhv = D.dhv[k];
    }
    LoopState S;
    if (REDUCED) S = *loop_of(P, L, ib);
    else S = step_state<T>(L, Lnext, mode);
    if (fix) {
        fix_advance<T, SPH>(P, E0, A, F, S, 0, t, ib);
        return;
    }
    if (!S.go) return;
    amr_update<T>(P, A, X, dh, dhu, dhv, S, 0, i, ib, t & 15, t >> 4);
}

// The corrector's fix-up and advance of the blocks that the stage left out.
template <class T, bool SPH>
__global__ __launch_bounds__(256) void k_amr_fix_advance(KParams P, StageIn<T> E0, AdvArgs<T> A, FluxOut<T> F,
                                                         DevLoop* L) {
    const int ib = ldu(P.fix, blockIdx.x);
    fix_advance<T, SPH>(P, E0, A, F, *loop_of(P, L, ib), 1, threadIdx.x, ib);
}

template <class T, bool SPH, bool FAST, int corr>
void stage(const KParams& P, const AmrBuffers<T>& B, const AdvArgs<T>& A, DevLoop* L, hipStream_t st) {
    T* h = const_cast<T*>(A.h);
    T* u = const_cast<T*>(A.u);
    T* v = const_cast<T*>(A.v);
    const FluxOut<T> F{B.Fhu, B.Fqux, B.Su, B.Fqvx, B.Fhv, B.Fqvy, B.Sv, B.Fquy};
    const Tend<T> D{B.dh, B.dhu, B.dhv};
    const dim3 quad((P.nblk + 3) / 4), blk(P.nblk), tpb(256);
    // With up to three levels the stage forms the halos itself: a block's prolongation depends on at
    // most its coarse neighbour's, which it evaluates again.  With more levels that chain is longer:
    // the halos are filled by a launch of their own and prolonged level by level, coarsest first.
    // So are they on meshes whose sides are no quadtree's (P.odd), which the recipes do not cover.
    const bool levels = P.wetdryfix && P.maxlevel - P.minlevel > 2;
    if (levels || P.odd) {
        const bool prolong = P.wetdryfix && P.maxlevel > P.minlevel;
        hipLaunchKernelGGL(k_amr_halo_refine<T>, blk, dim3(64), 0, st, P, h, u, v, B.zb, prolong ? B.hsnap : (T*)nullptr,
                           L, corr);
        for (int lev = P.minlevel + 2; prolong && lev <= P.maxlevel; lev++)
            hipLaunchKernelGGL(k_amr_prolong<T>, quad, tpb, 0, st, P, h, B.zb, (const T*)B.hsnap, lev, L, corr);
        hipLaunchKernelGGL((k_amr_stage<T, SPH, FAST, false, corr>), blk, tpb, 0, st, P, A, B.zb, F, D, L);
    } else {
        hipLaunchKernelGGL((k_amr_stage<T, SPH, FAST, true, corr>), blk, tpb, 0, st, P, A, B.zb, F, D, L);
    }
}

// Meshes of up to so many blocks have each workgroup of the predictor's advance
// work out the time step itself; larger ones, whose thousands of workgroups
// would repeat it, and batches, whose blocks are of many members, have it done
// by a launch in between.  A step with the launch and with the own reduction,
// two levels, us: 225 blocks FP32 32.3 and 31.4, FP64 34.9 and 34.2; 3,771
// blocks 91.3 and 90.8, 139.0 and 138.0; 6,989 blocks 142.6 and 142.0, 238.6
// and 237.6; 13,857 blocks 255.2 and 256.0, 490.4 and 490.5; 25,329 blocks
// 487.1 and 490.1, 918.8 and 917.9.  The line lies anywhere between 3,771 and
// 13,857 to within 1 us.
constexpr int SELF_REDUCE = 4096;

// Four launches: the predictor's stage, its advance, the corrector's stage with
// its advance, and the blocks whose faces wait for their finer neighbours'.
template <class T, bool SPH, bool FAST>
void amr_step(const KParams& P, const AmrBuffers<T>& B, DevLoop* L, DevLoop* Lnext, int advance_time, hipStream_t st,
              hipEvent_t* ev) {
    const dim3 blk(P.nblk), tpb(256);
    const FluxOut<T> F{B.Fhu, B.Fqux, B.Su, B.Fqvx, B.Fhv, B.Fqvy, B.Sv, B.Fquy};
    const Tend<T> D{B.dh, B.dhu, B.dhv};
    // the face fix-ups read the step-start state in both stages
    const StageIn<T> E0{B.h, B.u, B.v};
    if (!P.sid) launch_rain_now(P, L, st);  // batch members take no maps, rivers or level maps
    if (ev) (void)hipEventRecord(ev[0], st);
    // predictor: evolv_o = evolv + dt/2 L(evolv)
    const AdvArgs<T> a0{B.h, B.u, B.v, B.h, B.u, B.v, B.ho, B.uo, B.vo, B.zb, B.cf};
    stage<T, SPH, FAST, 0>(P, B, a0, L, st);
    if (ev) (void)hipEventRecord(ev[1], st);
    const bool reduce = P.sid || P.nblk > SELF_REDUCE;
    if (reduce) {
        if (P.sid) Lnext = L;
        launch_reduce_dt(sizeof(T) == 8 ? 0 : 1, L, Lnext, P.sid ? P.nmember : 1, advance_time, st);
    }
    if (ev) (void)hipEventRecord(ev[2], st);
    if (reduce)
        hipLaunchKernelGGL((k_amr_advance<T, SPH, true>), blk, tpb, 0, st, P, E0, a0, F, D, Lnext, Lnext, advance_time);
    else
        hipLaunchKernelGGL((k_amr_advance<T, SPH, false>), blk, tpb, 0, st, P, E0, a0, F, D, L, Lnext, advance_time);
    L = Lnext;  // the state past the reduction
    // corrector: evolv = friction(evolv + dt L(evolv_o)) + rain
    const AdvArgs<T> a1{B.ho, B.uo, B.vo, B.h, B.u, B.v, B.h, B.u, B.v, B.zb, B.cf};
    stage<T, SPH, FAST, 1>(P, B, a1, L, st);
    if (P.nfix > 0) hipLaunchKernelGGL((k_amr_fix_advance<T, SPH>), dim3(P.nfix), tpb, 0, st, P, E0, a1, F, L);
    if (ev) (void)hipEventRecord(ev[3], st);
}

template <class T, bool FAST>
void amr_step(const KParams& P, const void* buffers, DevLoop* L, DevLoop* Lnext, int advance_time, hipStream_t st,
              hipEvent_t* ev) {
    const AmrBuffers<T>& B = *(const AmrBuffers<T>*)buffers;
    // Cartesian grids: the metric terms are the constant 1 and their products fold away
    if (P.spherical) amr_step<T, true, FAST>(P, B, L, Lnext, advance_time, st, ev);
    else amr_step<T, false, FAST>(P, B, L, Lnext, advance_time, st, ev);
}

}  // namespace

void launch_amr_step(int precision, const KParams& P, const void* buffers, DevLoop* L, DevLoop* Lnext,
                     int advance_time, hipStream_t st, hipEvent_t* ev) {
    // BGF_FP32_FAST and BGF_FP32_COMP take the fast flux arithmetic (no compensated update here)
    if (precision == 0) amr_step<double, false>(P, buffers, L, Lnext, advance_time, st, ev);
    else if (precision == 1) amr_step<float, false>(P, buffers, L, Lnext, advance_time, st, ev);
    else amr_step<float, true>(P, buffers, L, Lnext, advance_time, st, ev);
}

__global__ __launch_bounds__(256) void k_amr_nbr(KParams P, int* nbr, int nbm) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b >= nbm) return;
    const int n[8] = {P.LeftBot[b], P.LeftTop[b], P.RightBot[b], P.RightTop[b],
                      P.BotLeft[b], P.BotRight[b], P.TopLeft[b], P.TopRight[b]};
    // the first-half neighbour arrays of the sides facing back: right, left, top, bottom
    const int* const back[4] = {P.RightBot, P.LeftBot, P.TopLeft, P.BotLeft};
    int info[8], flags = 0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const bool in = (unsigned)n[k] < (unsigned)nbm;  // unused slots may hold anything
        const int lev = in ? P.level[n[k]] : 0;
        const int bk = in && back[k >> 1][n[k]] == b ? 1 : 0;
        info[k] = (lev & 0xff) | (bk ? REC_BACK : 0);
        flags |= (in && lev > P.level[b] ? REC_FINER : 0) | (n[k] == b ? REC_EDGE : 0);
    }
#pragma unroll
    for (int k = 0; k < 8; k++) info[k] |= flags;
    int4* r = (int4*)(nbr + NBR * (size_t)b);
    r[0] = make_int4(n[0], n[1], n[2], n[3]);
    r[1] = make_int4(n[4], n[5], n[6], n[7]);
    r[2] = make_int4(info[0], info[1], info[2], info[3]);
    r[3] = make_int4(info[4], info[5], info[6], info[7]);
}

void launch_amr_nbr(const KParams& P, int* nbr, int nbm, int4* rcell, int2* rmeta, hipStream_t st) {
    if (nbm > 0) hipLaunchKernelGGL(k_amr_nbr, dim3((nbm + 255) / 256), dim3(256), 0, st, P, nbr, nbm);
    if (P.nblk > 0) hipLaunchKernelGGL(k_amr_recipes, dim3(P.nblk), dim3(192), 0, st, P, rcell, rmeta);
}

void launch_amr_fill(int precision, const KParams& P, void* z, hipStream_t st) {
    const dim3 quad((P.nblk + 3) / 4), tpb(256);
    if (precision == 0) hipLaunchKernelGGL(k_amr_fill<double>, quad, tpb, 0, st, P, (double*)z);
    else hipLaunchKernelGGL(k_amr_fill<float>, quad, tpb, 0, st, P, (float*)z);
}

void launch_amr_halo(int precision, const KParams& P, void* h, void* u, void* v, const void* zb, hipStream_t st) {
    const dim3 quad((P.nblk + 3) / 4), tpb(256);
    if (precision == 0)
        hipLaunchKernelGGL(k_amr_halo<double>, quad, tpb, 0, st, P, (double*)h, (double*)u, (double*)v,
                           (const double*)zb);
    else
        hipLaunchKernelGGL(k_amr_halo<float>, quad, tpb, 0, st, P, (float*)h, (float*)u, (float*)v,
                           (const float*)zb);
}

}  // namespace bgf
