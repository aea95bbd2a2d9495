// bgf_kernels.hip -- HIP/CDNA4 kernels of the BG_Flood Kurganov timestep on
// a one-level block-uniform grid.
//
// One workgroup of 256 threads (four wave64s) owns one 16x16 block; thread t
// owns cell (t % 16, t / 16).  Per step:
//
//   k_predictor  gathers h, zs = zb + h, u, v on a 20x20 tile (two cells of
//                each neighbour block, or the block's own edge cell at a
//                domain boundary) straight from the neighbours into LDS: the
//                halo fill of src/Halo.cu:586-616 plus the distance-2 reads of
//                gradientHalo (src/Gradients.cu:2713-3294) without a halo
//                pass.  It then forms the theta-minmod gradients
//                (src/Gradients.cu:921-957), the 17x16 X and 16x17 Y
//                Kurganov-Petrova faces (src/Kurganov.cu:474-641,
//                1404-1546), the tendencies with the wall patch folded in
//                (src/Advection.cu:160-254, src/Boundary.cu:587-760), and the
//                block's minimum CFL step (src/Advection.cu:470-498), which
//                it merges into one of 64 device slots with an atomic min.
//   k_corrector  works out dt from the slots (step_state: their minimum and
//                1/epsi, the 1.5x growth clamp and the output-time landing in
//                FP64, src/Advection.cu:511-535, then totaltime += dt,
//                src/Mainloop.cu:60; batches, whose blocks are of many members,
//                have k_reduce_dt do it once per member);
//                rebuilds U* = U + dt/2 L(U) (src/Advection.cu:332-385) on
//                its own 20x20 tile from U and the predictor tendencies, so
//                no U* array is written; forms the corrector fluxes of U*,
//                advances U^{n+1} = U + dt L(U*), applies bottom friction
//                (src/Friction.cu:89-148) and implicit rain
//                (src/Updateforcing.cu:530-581), and writes h, u, v to the
//                other buffer of a ping-pong pair.
//
// HBM traffic per cell-update: predictor reads h, u, v, zb and writes
// dh, dhu, dhv; corrector reads h, u, v, dh, dhu, dhv, zb, cf and writes
// h, u, v: 18 words.  Neighbour strips are re-read from cache.
//
// LDS holds array-of-structures quadruples, so a cell's state, a cell's
// gradients and a face's four fluxes are each one 16-byte (FP32) access.
//
// EXACT kernels (FAST = false) perform every operation of the reference CPU
// step in the same order and precision (this file is compiled with
// -ffp-contract=off; divisions and square roots round as IEEE's), so they
// reproduce the CPU step bit for bit.  FAST kernels use the hardware reciprocal
// and square root, fused multiply-adds, and carry the limited slopes as scaled
// half-cell increments: minmod(d1, (d1 + d2)/(2 theta), d2) of the raw
// differences, which (theta/2) times gives 0.5*minmod(theta d1, (d1 + d2)/2,
// theta d2); the factor theta/2 enters the reconstruction's multiply-adds.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdint.h>

#include <limits>

#include "bgf_common.h"

namespace bgf {

// src/Util_CPU.cu:243-263 without branches.  With d1 = theta*(s1-s0),
// d2 = (s2-s0)/2, d3 = theta*(s2-s1): s0 < s1 < s2 holds exactly when
// min(d1,d2,d3) > 0 (theta >= 1 and IEEE subtraction is zero only for equal
// operands), and then the reference returns that minimum; s0 > s1 > s2 holds
// exactly when max(d1,d2,d3) < 0 and then it returns that maximum; otherwise
// 0.  At most one of max(mn,0) and min(mx,0) is non-zero, so their sum is
// exact.
template <class T> __device__ __forceinline__ T minmod2c(T th, T half, T s0, T s1, T s2) {
    T d1 = th * (s1 - s0);
    T d2 = (s2 - s0) * half;
    T d3 = th * (s2 - s1);
    T mn = dmin(dmin(d1, d2), d3);
    T mx = dmax(dmax(d1, d2), d3);
    return dmax(mn, T(0.0)) + dmin(mx, T(0.0));
}

// Constants of the step in T, computed once on the host (make_cst) and
// passed by value, so kernels read them from scalar registers.
template <class T> struct Cst {
    T g, ga, CFL, theta, epsi, inv_epsi, eps_w, eps, delta, dxh, cmdinv, fc, cfl_delta, half;
    T th_s, mm_k;  // FAST slopes: half-cell increment = th_s * minmod(d1, mm_k (d1 + d2), d2)
    T sqg, src;    // FAST faces: sqrt(g); FAST source: -2 g th_s
    T mask, rain_step_scale;
    double eps_d, mask_d;
    FixedDiv<T> by_delta;
};

template <class T, bool FAST> Cst<T> make_cst(const KParams& P) {
    Cst<T> c;
    c.g = T(P.g);
    c.ga = c.g * T(0.5);
    c.CFL = T(P.CFL);
    c.theta = T(P.theta);
    c.epsi = sizeof(T) == 8 ? T(2.220446049250313e-16) : T(1.1920928955078125e-07);
    c.inv_epsi = T(1.0) / c.epsi;
    c.eps_w = T(P.eps) + c.epsi;
    c.eps = T(P.eps);
    c.eps_d = P.eps;
    c.delta = T(P.delta);
    c.dxh = c.delta * T(0.5);
    c.cmdinv = T(1.0) / (T(1.0) * c.delta);
    c.fc = T(P.fc);
    c.cfl_delta = c.CFL * c.delta;
    c.half = T(0.5);
    c.th_s = c.theta * T(0.5);
    // theta <= 0 limits every slope to zero, as minmod(theta d1, ., theta d2) does
    c.mm_k = c.th_s > T(0.0) ? T(0.25) / c.th_s : T(0.0);
    c.sqg = T(sqrt(P.g));
    c.src = T(-2.0) * c.g * c.th_s;
    c.mask = T(P.mask);
    c.mask_d = P.mask;
    c.rain_step_scale = T(0.0);
    c.by_delta = fixed_div(c.delta);
    return c;
}

// Hydrostatic reconstruction and central-upwind flux at one face between the
// "n" (left/bottom) cell and the "i" (right/top) cell, src/Kurganov.cu:62-164
// and 1865-1911.  Along Y the roles of u and v swap.  si/sn hold the cells'
// limited slopes of (h, zs, un, ut).  F: the mass flux, the normal-momentum
// flux that cell i takes and the one that cell n takes, the transverse flux.
// dt: the face's wave speed, 0 for a dry or still face; its CFL limit is
// cfl_delta / a (src/Kurganov.cu:102-105,159), and the block turns the largest
// speed into its step (cfl_delta / max a is min over faces of cfl_delta / a:
// rounded division is monotone).
template <class T, bool WANT_DT>
__device__ __forceinline__ bool kurg_face(const Cst<T>& C, const Q4<T>& qi, const Q4<T>& qn, const Q4<T>& si,
                                          const Q4<T>& sn, Q4<T>& F, T& dt) {
    const T hi = qi.a, hn = qn.a;
    const bool wet = hi > C.eps_w || hn > C.eps_w;
    const T zi = qi.b - hi;
    const T zn = qn.b - hn;
    const T dx = C.dxh;
    const T zl = zi - dx * (si.b - si.a);
    const T zr = zn + dx * (sn.b - sn.a);
    const T hl = hi - dx * si.a;
    const T up = qi.c - dx * si.c;
    const T hr = hn + dx * sn.a;
    const T um = qn.c + dx * sn.c;
    const T zlr = dmax(zl, zr);
    const T hp = dmax(T(0.0), hl + zl - zlr);
    const T hm = dmax(T(0.0), hr + zr - zlr);
    // KurgSolver
    const T cp = sqrt(C.g * hp);
    const T cmo = sqrt(C.g * hm);
    const T ap = dmax(dmax(up + cp, um + cmo), T(0.0));
    const T am = dmin(dmin(up - cp, um - cmo), T(0.0));
    const T qm = hm * um;
    const T qp = hp * up;
    const T a = dmax(ap, -am);
    const bool flow = a > C.epsi;
    const T ad = plain_rcp(ap - am);
    const T apm = ap * am;
    T fh = (ap * qm - am * qp + apm * (hp - hm)) * ad;
    T fu = (ap * (qm * um + C.ga * (hm * hm)) - am * (qp * up + C.ga * (hp * hp)) + apm * (qp - qm)) * ad;
    fh = flow ? fh : T(0.0);
    fu = flow ? fu : T(0.0);
    if (WANT_DT) dt = (flow && wet) ? a : T(0.0);
    const T fv = (fh > T(0.0) ? qn.d + C.dxh * sn.d : qi.d - C.dxh * si.d) * fh;
    const T sl = C.ga * (hp * hp - hl * hl + (hl + hi) * (zi - zl));
    const T sr = C.ga * (hm * hm - hr * hr + (hr + hn) * (zn - zr));
    F.a = wet ? fh : T(0.0);
    F.b = wet ? fu - sl : T(0.0);
    F.c = wet ? fu - sr : T(0.0);
    F.d = wet ? fv : T(0.0);
    return wet;
}

// The same face in the FAST kernels' arithmetic.  The tile carries the bed zb
// instead of zs (deviation form): the interface depths use zl - zr =
// (zb_i - zb_n) - (zi - zl) - (zr - zn), so no absolute elevation is rounded
// into a depth.  Slopes: h, un and ut over theta/2 (times C.th_s is the
// half-cell increment), and in .b the half-cell increment of the bed.
//
// With w = a+/(a+ - a-) and k = w a-, the central-upwind flux of a quantity
// with fluxes Fm, Fp and states Um, Up is Fp - w (Fp - Fm) + k (Up - Um).
// The gravity part of each momentum flux, g/2 hp^2, cancels against the same
// term of the hydrostatic source of the cell that takes it (src/Kurganov.cu:
// 132-145: g/2 (hp^2 - hl^2 + (hl + h) dz)), and what is left of a cell's two
// sources, g/2 (hl^2 - (hl + h) dz) - g/2 (hr^2 + (hr + h) dz), is -2 g h
// times the half-cell increment of zs, since hl and hr lie as far below and
// above h.  So a face keeps only F.b = up qp - w dF + k dq for cell i and
// F.c = F.b + g/2 (hp^2 - hm^2) for cell n, and the cell adds one term
// (cell_source), and no difference of squares of whole depths is rounded; where
// the water is at rest both parts are exactly zero.  With this and the exchange
// along x between lanes the FAST predictor issues 267 vector instructions a
// wave and block, 276 before, and 22 LDS instructions, 29 before.
template <bool WANT_DT>
__device__ __forceinline__ bool kurg_face_fast(const Cst<float>& C, const Q4<float>& qi, const Q4<float>& qn,
                                               const Q4<float>& si, const Q4<float>& sn, Q4<float>& F, float& dt) {
    const float th = C.th_s;
    const bool wet = fmaxf(qi.a, qn.a) > C.eps_w;
    const float hl = fmaf(-th, si.a, qi.a), up = fmaf(-th, si.c, qi.c);
    const float hr = fmaf(th, sn.a, qn.a), um = fmaf(th, sn.c, qn.c);
    const float dlr = (qi.b - qn.b) - si.b - sn.b;  // zl - zr
    const float hp = fmaxf(0.0f, hl + fminf(dlr, 0.0f));
    const float hm = fmaxf(0.0f, hr - fmaxf(dlr, 0.0f));
    const float sp = __builtin_amdgcn_sqrtf(hp), sm = __builtin_amdgcn_sqrtf(hm);
    const float ap = fmaxf(fmaxf(fmaf(C.sqg, sp, up), fmaf(C.sqg, sm, um)), 0.0f);
    const float am = fminf(fminf(fmaf(-C.sqg, sp, up), fmaf(-C.sqg, sm, um)), 0.0f);
    // both speeds zero (dry or still): the floor makes w and k zero, and the depths are zero too
    const float w = ap * __builtin_amdgcn_rcpf(fmaxf(ap - am, 1e-30f));
    const float k = w * am;
    const float qp = hp * up, qm = hm * um;
    const float dq = qp - qm, dh = hp - hm;
    const float fh = fmaf(k, dh, fmaf(-w, dq, qp));
    const float mp = qp * up;
    const float g0 = dh * (hp + hm);
    const float dF = fmaf(C.ga, g0, fmaf(-qm, um, mp));
    const float fp = fmaf(k, dq, fmaf(-w, dF, mp));
    const float fm = fmaf(C.ga, g0, fp);
    if (WANT_DT) dt = wet ? fmaxf(ap, -am) : 0.0f;
    F.a = wet ? fh : 0.0f;
    F.b = wet ? fp : 0.0f;
    F.c = wet ? fm : 0.0f;
    F.d = (F.a > 0.0f ? fmaf(th, sn.d, qn.d) : fmaf(-th, si.d, qi.d)) * F.a;
    return wet;
}

// A cell's hydrostatic source along one direction, per cell size: what
// kurg_face_fast leaves out of its two faces, taken with the left (bottom)
// face's momentum flux, which only this cell reads; so a wall, where the cell
// takes no difference, drops it too.  gzs, gh: the cell's slopes of zs and h
// over theta/2; hb, ha: the depths of the cells before and after it.  A face is wet if
// either of its cells is, so a wet cell has both; a dry one takes the part of
// each wet neighbour's face.
__device__ __forceinline__ float cell_source(const Cst<float>& C, float h, float gzs, float gh, float hb, float ha) {
    float s = C.src * h * gzs;
    if (!(h > C.eps_w)) {
        const float a = C.th_s * gh, dz = C.th_s * (gzs - gh);
        const float hl = h - a, hr = h + a;
        const float xl = hb > C.eps_w ? fmaf(hl, hl, -(hl + h) * dz) : 0.0f;
        const float yr = ha > C.eps_w ? fmaf(hr, hr, (hr + h) * dz) : 0.0f;
        s = C.ga * (xl - yr);
    }
    return s;
}

// The block in LDS.  ROW (the FAST kernels): along x the neighbours come from
// the lanes beside, and only the ends of the rows pass through here.  The
// faces take the slopes' place once every thread has formed its own.
template <class T, bool ROW> struct Tile {
    Q4<T> q[20 * TP];   // (h, zs, u, v) at x, y in [-2, 17], corners unused
    union {
        struct {
            Q4<T> gy[18 * GYP];             // slopes along y of (h, zs, v, u) at x in [0,15], y in [-1,16]
            Q4<T> gx[ROW ? 1 : 16 * GXP];   // slopes along x of (h, zs, u, v) at x in [-1,16], y in [0,15]
        };
        struct {
            Q4<T> fy[17 * BW];              // (Fhv, Fqvy, Sv, Fquy) at Y faces, x in [0,15], yf in [0,16]
            Q4<T> fx[ROW ? 1 : 16 * FP];    // (Fhu, Fqux, Su, Fqvx) at X faces, xf in [0,16]
        };
    };
    Q4<T> gxr[ROW ? 2 * BW : 1];  // ROW: slopes along x at x = -1, then at x = 16
    Q4<T> gxe[ROW ? BW : 1];      // ROW: and at x = 15
    Q4<T> fe[ROW ? BW : 1];       // ROW: X faces at xf = 16
    T red[4];
    int next[4];  // queue positions: slot j & 3 holds position j
};

// Strip slot k in [0, 128): waves 0 and 1 fetch the two-deep x strips (left,
// right) and y strips (bottom, top) of the 20x20 tile.  strip_cell gives the
// tile position.
__device__ __forceinline__ int strip_off(int k) {
    const int s = (k >> 4) & 3;  // 0: -1, 1: -2, 2: 16, 3: 17
    return s < 2 ? -1 - s : 14 + s;
}
__device__ __forceinline__ int strip_cell(int k) {
    const int j = k & 15, o = strip_off(k);
    return k < 64 ? tix(o, j) : tix(j, o);
}

// The strip sources in a form that costs a few vector instructions per block:
// a strip slot k < 128 always reads from the same side (k / 32: left, right,
// bottom, top), and its source cell's position inside the source block takes
// one of two values fixed per slot, the neighbour's cell or, without a
// neighbour (the neighbour index is the block itself), the block's own edge
// cell.  Both are formed once per thread as byte offsets, packed in one
// register per layout (the neighbour's cell in the low 16 bits, the own edge
// cell in the high 16 bits; offsets within a block are below 2^16): kb in the
// block layout, ki in the interior layout.  Per block the source block is the
// side's neighbour index in either case.
struct StripK {
    unsigned kb, ki;
};
template <class T> __device__ __forceinline__ StripK strip_k(int k) {
    const int j = k & 15, o = strip_off(k);
    const bool lo = o < 0, isx = k < 64;
    const int an = lo ? BW + o : o - BW;   // along the normal, in the neighbour
    const int as = lo ? 0 : BW - 1;        // along the normal, in the block itself
    const int xn = isx ? an : j, yn = isx ? j : an;
    const int xs = isx ? as : j, ys = isx ? j : as;
    StripK r;
    r.kb = (unsigned)memloc(xn, yn, 0) * sizeof(T) | ((unsigned)memloc(xs, ys, 0) * sizeof(T)) << 16;
    r.ki = (unsigned)(yn * BW + xn) * sizeof(T) | ((unsigned)(ys * BW + xs) * sizeof(T)) << 16;
    return r;
}
// The offset of a packed pair: the own edge cell's if self, else the neighbour's.
__device__ __forceinline__ unsigned strip_pick(unsigned packed, bool self) {
    return __builtin_amdgcn_ubfe(packed, self ? 16u : 0u, 16u);
}
// Source block of thread t's strip slot (t < 128): waves 0 and 1 hold the x
// and y strips, lanes 0-31 the low side and 32-63 the high side.
__device__ __forceinline__ int strip_block(int t, int nL, int nR, int nB, int nT) {
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int na = w == 0 ? nL : nB, nc = w == 0 ? nR : nT;
    return (t & 32) ? nc : na;
}

// FAST minmod of three: minmod(d1, d2, d3) = med3(d1, med3(d2, d3, 0), 0)
// (two operands of one sign give their smaller magnitude, mixed signs give
// 0), two v_med3_f32 instead of min3, max3, max, min and add.  Equal to
// minmod2c for every non-NaN input up to the sign of a zero result.
__device__ __forceinline__ float minmod3f(float d1, float d2, float d3) {
    return __builtin_amdgcn_fmed3f(d1, __builtin_amdgcn_fmed3f(d2, d3, 0.0f), 0.0f);
}
// minmod2c(theta, 1/2, s0, s1, s2) / theta, with k = 1/(2 theta).
__device__ __forceinline__ float minmod2f(float k, float s0, float s1, float s2) {
    return minmod3f(s1 - s0, (s2 - s0) * k, s2 - s1);
}
// minmod2f of the sums z + h from the differences of each part: the slope of
// zs = zb + h without forming zs, whose FP32 rounding (ulp of the bed
// elevation) would swamp millimetre depths (deviation form).
__device__ __forceinline__ float minmod2sf(float k, float z0, float z1, float z2, float h0, float h1, float h2) {
    return minmod3f((z1 - z0) + (h1 - h0), ((z2 - z0) + (h2 - h0)) * k, (z2 - z1) + (h2 - h1));
}

// Slopes of (h, zs, u, v) of cell c between m and p; in FAST kernels those of
// h, u and v over theta/2 and in .b the half-cell increment of the bed, with
// the slope of zs over theta/2 in gzs.
template <class T, bool FAST>
__device__ __forceinline__ Q4<T> slopes(const Cst<T>& C, const Q4<T>& m, const Q4<T>& c, const Q4<T>& p, T& gzs) {
    Q4<T> g;
    if constexpr (FAST) {
        static_assert(sizeof(T) == 4, "FAST kernels are FP32");
        g.a = minmod2f(C.mm_k, m.a, c.a, p.a);
        gzs = minmod2sf(C.mm_k, m.b, c.b, p.b, m.a, c.a, p.a);
        g.b = C.th_s * (gzs - g.a);
        g.c = minmod2f(C.mm_k, m.c, c.c, p.c);
        g.d = minmod2f(C.mm_k, m.d, c.d, p.d);
    } else {
        g.a = minmod2c(C.theta, C.half, m.a, c.a, p.a);
        g.b = minmod2c(C.theta, C.half, m.b, c.b, p.b);
        g.c = minmod2c(C.theta, C.half, m.c, c.c, p.c);
        g.d = minmod2c(C.theta, C.half, m.d, c.d, p.d);
        g = div4(C.by_delta, g);
    }
    return g;
}

// Extra work of a tile beyond one cell per thread goes to distinct waves, each
// as one section with its lanes filled: the 64 halo-ring slopes to wave 2
// and the 32 seventeenth faces to wave 3 (waves 0 and 1 fetch the strips, and
// in the corrector also advance them).

// Values of the lanes beside a lane in its row of 16 (the cells beside it along
// x), through the data-parallel primitives of the vector ALU: from_left gives
// each lane the value of the lane before it, and lane 0 of the row its `end`;
// from_right that of the lane after it, and lane 15 its `end`.
template <int CTRL> __device__ __forceinline__ int dpp_move(int end, int v) {
    return __builtin_amdgcn_update_dpp(end, v, CTRL, 0xf, 0xf, false);
}
template <int CTRL> __device__ __forceinline__ float dpp_move(float end, float v) {
    return __int_as_float(dpp_move<CTRL>(__float_as_int(end), __float_as_int(v)));
}
template <int CTRL> __device__ __forceinline__ double dpp_move(double end, double v) {
    return __hiloint2double(dpp_move<CTRL>(__double2hiint(end), __double2hiint(v)),
                            dpp_move<CTRL>(__double2loint(end), __double2loint(v)));
}
constexpr int ROW_SHR1 = 0x111, ROW_SHL1 = 0x101;
template <class T> __device__ __forceinline__ T from_left(T end, T v) { return dpp_move<ROW_SHR1>(end, v); }
template <class T> __device__ __forceinline__ T from_right(T end, T v) { return dpp_move<ROW_SHL1>(end, v); }
template <class T> __device__ __forceinline__ Q4<T> from_left(const Q4<T>& e, const Q4<T>& v) {
    return Q4<T>{from_left(e.a, v.a), from_left(e.b, v.b), from_left(e.c, v.c), from_left(e.d, v.d)};
}
template <class T> __device__ __forceinline__ Q4<T> from_right(const Q4<T>& e, const Q4<T>& v) {
    return Q4<T>{from_right(e.a, v.a), from_right(e.b, v.b), from_right(e.c, v.c), from_right(e.d, v.d)};
}

// Slopes of the tile: every thread its own cell along x and y (gzx, gzy: those
// of zs in FAST kernels); the halo ring on wave 2, lanes 0-31 the x slopes at
// x = -1, 16 and lanes 32-63 the y slopes at y = -1, 16.  qh (FAST): lanes 0-7
// of a row hold its halo cell at x = -1, lanes 8-15 that at x = 16.
template <class T, bool FAST>
__device__ __forceinline__ void tile_gradients(Tile<T, FAST>& s, const Cst<T>& C, int t, const Q4<T>& q, Q4<T>& gxo,
                                               Q4<T>& gyo, T& gzx, T& gzy) {
    {
        const int x = t & 15, y = t >> 4;
        const int c = tix(x, y);
        if constexpr (FAST) {
            const Q4<T> qh = s.q[tix(x < BW / 2 ? -1 : BW, y)];
            gxo = slopes<T, FAST>(C, from_left(qh, q), q, from_right(qh, q), gzx);
            if (x == BW - 1) s.gxe[y] = gxo;
        } else {
            gxo = slopes<T, FAST>(C, s.q[c - 1], q, s.q[c + 1], gzx);
            s.gx[gxi(x, y)] = gxo;
        }
        Q4<T> g = slopes<T, FAST>(C, s.q[c - TP], q, s.q[c + TP], gzy);
        // y slopes stored as (h, zs, v, u)
        gyo.a = g.a; gyo.b = g.b; gyo.c = g.d; gyo.d = g.c;
        s.gy[gyi(x, y)] = gyo;
    }
    if ((t >> 6) == 2) {
        const int r = t & 63, j = r & 15;
        const bool isx = r < 32;
        const int o = (r & 16) ? BW : -1;
        const int c = isx ? tix(o, j) : tix(j, o);
        const int d = isx ? 1 : TP;
        T gz;
        const Q4<T> g = slopes<T, FAST>(C, s.q[c - d], s.q[c], s.q[c + d], gz);
        Q4<T> gs;
        gs.a = g.a; gs.b = g.b; gs.c = isx ? g.c : g.d; gs.d = isx ? g.d : g.c;
        *(isx ? (FAST ? &s.gxr[r] : &s.gx[gxi(o, j)]) : &s.gy[gyi(j, o)]) = gs;
    }
}

template <class T, bool FAST, bool WANT_DT>
__device__ __forceinline__ bool face(const Cst<T>& C, const Q4<T>& qi, const Q4<T>& qn, const Q4<T>& si,
                                     const Q4<T>& sn, Q4<T>& F, T& dt) {
    bool wet;
    if constexpr (FAST) wet = kurg_face_fast<WANT_DT>(C, qi, qn, si, sn, F, dt);
    else wet = kurg_face<T, WANT_DT>(C, qi, qn, si, sn, F, dt);
    finish(F);
    return wet;
}
template <class T> __device__ __forceinline__ Q4<T> swap_uv(const Q4<T>& q) { return Q4<T>{q.a, q.b, q.d, q.c}; }

// Fluxes of the tile state and the tendencies of the thread's cell, with the
// wall patch (noslipbndQ, src/Boundary.cu:1887-1891) applied as operand
// substitutions: at a left (bottom) wall the boundary face has no mass flux
// and the first cell's right-face source S is replaced by its left-face Fq;
// at a right (top) wall the boundary face has no mass flux and the last
// cell's left-face Fq is replaced by its right-face S.  Either way the cell
// takes no normal-momentum difference.  Returns the wave speed that limits the
// cell's dtmax (0: none), see kurg_face.  q is the state the thread stored for
// its cell; it, the cell's slopes and its left and bottom faces stay in
// registers.  FAST kernels exchange along x between lanes: with every exchange
// through LDS the FAST predictor's 30 accesses of 16 bytes a lane, with their
// bank conflicts, took all of its 655 us at 8192 x 8192 cells, 21 accesses and
// 28 more vector instructions 622.  The exact FP32 kernels need 41 of their 48
// us (1520 x 2032 cells) to issue vector instructions at the top clock of 2.4
// GHz and gain nothing from that trade.
template <class T> struct CellFaces {
    Q4<T> l, r, b, t;
};
template <class T, bool FAST, bool WANT_DT>
__device__ __forceinline__ T tile_fluxes(Tile<T, FAST>& s, const Cst<T>& C, int t, const Q4<T>& q, bool wl, bool wr,
                                         bool wb, bool wt, CellFaces<T>& A, T& dh, T& dhu, T& dhv) {
    Q4<T> gx, gy;
    T gzx = T(0), gzy = T(0);
    tile_gradients<T, FAST>(s, C, t, q, gx, gy, gzx, gzy);
    __syncthreads();
    const int x = t & 15, y = t >> 4;
    const int ci = tix(x, y);
    T dtx = T(0.0), dty = T(0.0), dtd;  // wave speeds of the cell's faces
    Q4<T> Fl, Fb, Fe;
    if constexpr (FAST) {
        const Q4<T> qh = s.q[tix(x < BW / 2 ? -1 : BW, y)];
        face<T, FAST, WANT_DT>(C, q, from_left(qh, q), gx, from_left(s.gxr[y], gx), Fl, dtx);
        Fl.b += cell_source(C, q.a, gzx, gx.a, from_left(qh.a, q.a), from_right(qh.a, q.a));
    } else {
        face<T, FAST, WANT_DT>(C, q, s.q[ci - 1], gx, s.gx[gxi(x - 1, y)], Fl, dtx);
    }
    const Q4<T> qb = s.q[ci - TP];
    const bool wy = face<T, FAST, WANT_DT>(C, swap_uv(q), swap_uv(qb), gy, s.gy[gyi(x, y - 1)], Fb, dty);
    if constexpr (FAST) Fb.b += cell_source(C, q.a, gzy, gy.a, qb.a, s.q[ci + TP].a);
    const bool edge = t >= 192 && t < 224, ex = t < 208;
    if (edge) {
        // the seventeenth faces on wave 3: lanes 0-15 the X faces at xf = 16,
        // lanes 16-31 the Y faces at yf = 16
        const int j = t & 15;
        const int ce = ex ? tix(BW, j) : tix(j, BW);
        Q4<T> qi = s.q[ce], qn = s.q[ce - (ex ? 1 : TP)];
        if (!ex) {
            qi = swap_uv(qi);
            qn = swap_uv(qn);
        }
        const Q4<T>* gi = ex ? (FAST ? &s.gxr[BW + j] : &s.gx[gxi(BW, j)]) : &s.gy[gyi(j, BW)];
        const Q4<T>* gn = ex ? (FAST ? &s.gxe[j] : &s.gx[gxi(BW - 1, j)]) : &s.gy[gyi(j, BW - 1)];
        face<T, FAST, false>(C, qi, qn, *gi, *gn, Fe, dtd);
    }
    __syncthreads();  // the slopes are read: the faces take their place
    s.fy[t] = Fb;
    if (!FAST) s.fx[y * FP + x] = Fl;
    if (edge) *(!ex ? &s.fy[BW * BW + (t & 15)] : FAST ? &s.fe[t & 15] : &s.fx[(t & 15) * FP + BW]) = Fe;
    // The cell's limiting speed: its X face then its Y face, a dry Y face storing 1/epsi outright
    // (src/Kurganov.cu:1488-1491), i.e. no limit; 1/epsi caps the step at the reduction.
    T dtc = T(0.0);
    if (WANT_DT) dtc = wy ? dmax(dtx, dty) : T(0.0);
    __syncthreads();
    Q4<T> Fr;
    if constexpr (FAST) Fr = from_right(s.fe[y], Fl);
    else Fr = s.fx[y * FP + x + 1];
    const Q4<T> Ft = s.fy[t + BW];
    A = CellFaces<T>{Fl, Fr, Fb, Ft};
    T Fhl = Fl.a, Fhr = Fr.a, Fql = Fl.b, Sr = Fr.c;
    T Fhb = Fb.a, Fht = Ft.a, Fqb = Fb.b, St = Ft.c;
    if (wl && x == 0) { Fhl = T(0.0); Sr = Fql; }
    if (wr && x == BW - 1) { Fhr = T(0.0); Fql = Sr; }
    if (wb && y == 0) { Fhb = T(0.0); St = Fqb; }
    if (wt && y == BW - 1) { Fht = T(0.0); Fqb = St; }
    // src/Advection.cu:236-250 (Cartesian: the metric terms vanish)
    dh = T(-1.0) * (Fhr - Fhl + Fht - Fhb) * C.cmdinv;
    if (FAST) {
        dhu = ((Fql - Sr) + (Fb.d - Ft.d)) * C.cmdinv + C.fc * q.a * q.d;
        dhv = ((Fqb - St) + (Fl.d - Fr.d)) * C.cmdinv - C.fc * q.a * q.c;
    } else {
        dhu = (Fql + Fb.d - Sr - Ft.d) * C.cmdinv + C.fc * q.a * q.d;
        dhv = (Fqb + Fl.d - St - Fr.d) * C.cmdinv - C.fc * q.a * q.c;
    }
    return dtc;
}

// Tendencies of an edge cell of a block on a side of type 2 or 3, recomputed
// from its faces A with the boundary face's mass flux from bnd_flux, or the
// no-slip patch on a dry face.  Runs only for blocks with such a side, after
// tile_fluxes; q: the cell's stage state.
template <class T, bool FAST>
__device__ __forceinline__ void open_sides(const CellFaces<T>& A, const Q4<T>& q, const Cst<T>& C, const KParams& P, int t, int ib, int nL, int nR, int nB,
                           int nT, double tstage, const T* h, const T* u, const T* v, const T* zb, T& dh, T& dhu,
                           T& dhv) {
    const int x = t & 15, y = t >> 4;
    const int bt = blk_btype(P, ib);
    if (bt < 2) return;
    const int side[4] = {nL == ib && x == 0 ? bt : -1, nR == ib && x == BW - 1 ? bt : -1,
                         nB == ib && y == 0 ? bt : -1, nT == ib && y == BW - 1 ? bt : -1};
    if (side[0] < 2 && side[1] < 2 && side[2] < 2 && side[3] < 2) return;
    const BSeg& S = P.seg[P.bseg[ib]];
    T F[4] = {A.l.a, A.r.a, A.b.a, A.t.a};
    bool slip[4];
#pragma unroll
    for (int sd = 0; sd < 4; sd++) {
        slip[sd] = side[sd] == 0;
        if (side[sd] >= 2) {
            const int ci = sd == 0 ? memloc(0, y, ib) : sd == 1 ? memloc(BW - 1, y, ib) : sd == 2 ? memloc(x, 0, ib)
                                                                                            : memloc(x, BW - 1, ib);
            const int cin = sd == 0 ? memloc(1, y, ib) : sd == 2 ? memloc(x, 1, ib) : ci;
            const T hi = h[ci], hin = h[cin];
            T q = F[sd];
            // the face's position: ix = 0 or 16 across the block, the cell's along it
            const int fx = sd == 0 ? 0 : sd == 1 ? BW : x, fy = sd == 2 ? 0 : sd == 3 ? BW : y;
            if (bnd_flux<T>(P, sd, side[sd], seg_level<T>(P, S, tstage, ib, fx, fy), bnd_taper<T>(P, S, tstage),
                            zb[ci] + hi, hi, zb[cin] + hin, hin, (sd < 2 ? u : v)[cin], q))
                F[sd] = q;
            else
                slip[sd] = true;
        }
        if (slip[sd]) F[sd] = T(0.0);
    }
    dh = T(-1.0) * (F[1] - F[0] + F[3] - F[2]) * C.cmdinv;
    // the no-slip patch leaves no normal-momentum difference (in FAST kernels no source either)
    if ((side[0] >= 2 && slip[0]) || (side[1] >= 2 && slip[1])) {
        const T lo = A.l.b, hi = A.r.c, Fq = FAST ? T(0.0) : slip[1] ? hi : lo;
        dhu = (Fq + A.b.d - Fq - A.t.d) * C.cmdinv + C.fc * q.a * q.d;
    }
    if ((side[2] >= 2 && slip[2]) || (side[3] >= 2 && slip[3])) {
        const T lo = A.b.b, hi = A.t.c, Fq = FAST ? T(0.0) : slip[3] ? hi : lo;
        dhv = (Fq + A.l.d - Fq - A.r.d) * C.cmdinv - C.fc * q.a * q.c;
    }
}

// src/Advection.cu:332-385.  The drying limiter evaluates
// min(dt, max(h, eps)/|dh|) in double precision in the reference.
// FAST: the limiter without its division.  It binds where dt |dh| > m =
// max(h, eps) with dh < 0; then edt = m / |dh| and the new depth is h - m (0 for
// a wet cell), at most eps, where u and v are set to 0 whatever edt is; where it
// does not bind edt = dt.  So the depth is h - m or h + dt dh, and the momentum
// uses dt.
template <class T> __device__ __forceinline__ bool dry_limit(const Cst<T>& C, int fmc, T dt, T hold, T dhi, T& m) {
    m = dmax(hold, C.eps);
    return !fmc && fma(dt, dhi, m) < T(0.0);
}

template <class T, bool FAST>
__device__ __forceinline__ void advance(const Cst<T>& C, int fmc, T dt, T hold, T uold, T vold, T dhi, T dhui, T dhvi,
                                        T& ho, T& uo, T& vo) {
    typedef Ar<T, FAST> A;
    if (FAST) {
        T m;
        const bool lim = dry_limit(C, fmc, dt, hold, dhi, m);
        ho = lim ? hold - m : fma(dt, dhi, hold);
        T r = A::rcp(ho);
        uo = ho > C.eps ? fma(hold, uold, dt * dhui) * r : T(0.0);
        vo = ho > C.eps ? fma(hold, vold, dt * dhvi) * r : T(0.0);
        return;
    }
    const T edt = fmc ? dt : dry_step(dt, hold, dhi, C.eps, C.eps_d);
    ho = hold + edt * dhi;
    if (ho > C.eps) {
        uo = (hold * uold + edt * dhui) / ho;
        vo = (hold * vold + edt * dhvi) / ho;
    } else {
        uo = T(0.0);
        vo = T(0.0);
    }
}


// Workgroups are dispatched round-robin over the eight XCDs (NXCD), each with
// its own L2: the persistent kernels give each XCD a contiguous range of
// blocks so a block's neighbours are mostly fetched into the same L2.

// A value that every lane holds, kept in scalar registers.
__device__ __forceinline__ float uniform(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}
__device__ __forceinline__ double uniform(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}
// Cell k of block ib of array a: the array base (a kernel argument, in scalar
// registers for the whole launch) plus one 32-bit byte offset per thread that
// carries both the block and the cell, boff(ib) + k * sizeof(T), so each load
// is a saddr + voffset access with no 64-bit address arithmetic.  Per block the
// scalar state is the block index alone and the offset costs one vector add
// per array layout; forming a 64-bit block base per array in scalar registers
// instead (two per array and block, with the next block's prefetch in flight)
// outgrows the scalar register file and spills.  The empty asm in vof keeps the
// offset a 32-bit vector value beside each access (the compiler would otherwise
// widen it into 64-bit per-array addresses).  Byte offsets stay below 2^32:
// check_param limits nblkmem * 324 * sizeof(T).
typedef __attribute__((address_space(1))) char gchar;
__device__ __forceinline__ unsigned vof(unsigned kb) {
    asm("" : "+v"(kb));
    return kb;
}
template <class T> __device__ __forceinline__ unsigned boff(int ib) { return (unsigned)ib * (unsigned)(BS * sizeof(T)); }
template <class T> __device__ __forceinline__ unsigned boff_i(int ib) {
    return (unsigned)ib * (unsigned)(BSI * sizeof(T));
}
template <class T> __device__ __forceinline__ T ldo(const T* a, unsigned off) {
    return *(const __attribute__((address_space(1))) T*)((const gchar*)a + vof(off));
}
template <class T> __device__ __forceinline__ void sto(T* a, unsigned off, T v) {
    *(__attribute__((address_space(1))) T*)((gchar*)a + vof(off)) = v;
}
template <class T> __device__ __forceinline__ T ldno(const T* a, unsigned off) {
    return __builtin_nontemporal_load((const __attribute__((address_space(1))) T*)((const gchar*)a + vof(off)));
}
template <class T> __device__ __forceinline__ void stno(T* a, unsigned off, T v) {
    __builtin_nontemporal_store(v, (__attribute__((address_space(1))) T*)((gchar*)a + vof(off)));
}

struct Nb {
    int ib, nL, nR, nB, nT, sid;
};
// The block at position pos of the processing order with its neighbours and
// member, one 32-byte scalar load of the position's record (launch_records).
typedef int Rec8 __attribute__((ext_vector_type(8)));
template <bool BATCH> __device__ __forceinline__ Nb block_nb(const KParams& P, int pos) {
    const Rec8 r = ((const __attribute__((address_space(4))) Rec8*)P.rec)[pos];
    Nb n;
    n.ib = r[0];
    n.nL = r[1];
    n.nR = r[2];
    n.nB = r[3];
    n.nT = r[4];
    n.sid = BATCH ? r[5] : 0;
    return n;
}

__global__ __launch_bounds__(256) void k_records(KParams P, int* rec) {
    const int k = blockIdx.x * 256 + threadIdx.x;
    if (k >= P.nblk) return;
    const int ib = P.order[k];
    int4* r = (int4*)(rec + 8 * (size_t)k);
    r[0] = make_int4(ib, P.LeftBot[ib], P.RightBot[ib], P.BotLeft[ib]);
    r[1] = make_int4(P.TopLeft[ib], P.sid ? P.sid[ib] : 0, 0, 0);
}

void launch_records(const KParams& P, int* rec, hipStream_t st) {
    if (P.nblk > 0) hipLaunchKernelGGL(k_records, dim3((P.nblk + 255) / 256), dim3(256), 0, st, P, rec);
}

// The CFL step of cells whose largest limiting wave speed is smax: cfl_delta /
// smax, which equals the minimum over their faces of the reference's
// cfl_delta / a (a correctly rounded division is monotone in a), or 1/epsi
// where no face limits it.
template <class T, bool FAST> __device__ __forceinline__ T speed_dt(const Cst<T>& C, T smax) {
    if (!(smax > T(0.0))) return C.inv_epsi;
    const T d = FAST ? C.cfl_delta * Ar<T, FAST>::rcp(smax) : C.cfl_delta / smax;
    return d < C.inv_epsi ? d : C.inv_epsi;
}

// Merges a member's partial maximum speed into its dt slots: one atomic per
// wave, no workgroup barrier (members change often along a workgroup's blocks).
template <class T, bool FAST> __device__ __forceinline__ void wave_flush(const Cst<T>& C, DevLoop* L, T v, int t) {
    for (int off = 32; off > 0; off >>= 1) v = dmax(v, __shfl_xor(v, off, 64));
    if ((t & 63) == 0) slot_min(L, (blockIdx.x << 2) + (t >> 6), speed_dt<T, FAST>(C, v));
}

// Persistent workgroups take their blocks from a queue per XCD: the XCD's
// contiguous range of the processing order is handed out one position at a
// time by an atomic counter, so the blocks in flight on an XCD always form a
// compact window of consecutive positions (whose neighbour strips are then
// in that XCD's L2), however unevenly the workgroups progress.  A static
// stride lets the workgroups drift apart over a launch and the window widen
// beyond what L2 holds.
//
// queue[x * QSTRIDE] (x < 8) are the predictor's counters and
// queue[(8 + x) * QSTRIDE] the corrector's, each in a line of its own.
// Each kernel, when it runs, zeroes the other kernel's counters (the other
// kernel is not running: both are on one stream), so every launch finds its
// own at zero: the first launch from the allocation, later ones from the
// other kernel's launch in between (the zeroing comes before a kernel's
// early return, and a launch that returns early takes no position).
// A workgroup's first position is its rank on the XCD, and the queue hands out
// those after the workgroups' first ones; where the XCD's range has no more
// (more false: a domain of up to about 1,500 blocks) nothing is taken.
//
// Queue positions.  Each workgroup's positions increase (one thread's
// atomics on one counter are ordered), so the first one past the range ends
// the walk and no position is lost; the workgroup reads position j from slot
// j & 3 of the tile after a barrier.
//
// Predictor: thread 0 takes position j + 1 into its slot in front of the
// barrier of iteration j, waiting for the atomic there (queue_take_now).
// Corrector: thread 0 holds in `pend` the value of an atomic issued one
// iteration earlier; queue_publish writes it as position j and issues the
// atomic for position j + 1, so nothing waits for the atomic's round trip
// (nor, since stores share its counter, for the previous block's stores) in
// front of the barrier.  Measured on the 8192^2 rain workload the deferred
// form takes 1.8 % off the corrector and adds 3 % to the predictor, hence the
// split.  A slot is rewritten at least two iterations after it was read.
__device__ __forceinline__ void queue_take_now(int* q, int start, int* next, int j, int t) {
    if (t == 0) next[j & 3] = start + __hip_atomic_fetch_add(q, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int queue_take(int* q) {
    // A zero offset the compiler cannot see through makes the address
    // divergent, which keeps this a plain one-lane atomic: the wave-level
    // rewrite of a uniform-address atomic broadcasts the result right after
    // it and so would wait for its round trip on the spot.
    int z = 0;
    asm volatile("" : "+v"(z));
    return __hip_atomic_fetch_add(q + z, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void queue_publish(int* q, int start, int* next, int j, int t, int& pend) {
    if (t == 0) {
        next[j & 3] = start + pend;
        pend = queue_take(q);
    }
}
// The last atomic's value is not used: wait for it before the wave ends.
__device__ __forceinline__ void queue_end(int t, int pend) {
    if (t == 0) asm volatile("" ::"v"(pend));
}
__device__ __forceinline__ int queue_read(const int* next, int j) {
    return __builtin_amdgcn_readfirstlane(next[j & 3]);
}

// Persistent predictor: each workgroup walks its block sequence, prefetching
// the next block's cells into registers while the current block is computed
// from the LDS tile, so the gathers of one block overlap the arithmetic of the
// previous one.  One atomic min per workgroup (per member and workgroup in a
// batch, whose processing order keeps each member's blocks together; blocks
// of members that reached their end time are skipped).
// EXT kernels also take the open boundaries (types 2, 3), rivers and rain maps;
// the plain ones leave that code out, which keeps their register count (and
// so their occupancy) down.
template <class T, bool FAST, bool BATCH, bool DEV, bool EXT = false>
__global__ __launch_bounds__(256) void k_predictor(KParams P, Cst<T> C, StepBuffers<T> B, DevLoop* L) {
    if (blockIdx.x == 0 && threadIdx.x < NXCD) P.queue[(NXCD + threadIdx.x) * QSTRIDE] = 0;  // the corrector's
    if (!BATCH && L->done) return;
    __shared__ Tile<T, FAST> s;
    const int t = threadIdx.x;
    const int x = t & 15, y = t >> 4;
    const int xcd = blockIdx.x % NXCD;
    const Range R = xcd_range(xcd, P.nblk);
    int* const qc = P.queue + xcd * QSTRIDE;
    const int cs = strip_cell(t);
    const StripK sk = strip_k<T>(t);
    T smax = T(0.0);  // the largest limiting wave speed of the workgroup's cells so far
    int csid = -1;
    T ph = T(0), pz = T(0), pu = T(0), pv = T(0), sh = T(0), sz = T(0), su = T(0), sv = T(0);
    const unsigned kb = (unsigned)memloc(x, y, 0) * sizeof(T);
    const unsigned ki = (unsigned)(y * BW + x) * sizeof(T);  // in the tendency arrays
    auto fetch = [&](const Nb& n) {
        const unsigned o = boff<T>(n.ib) + kb;
        ph = ldo(B.h, o); pz = ldo(B.zb, o); pu = ldo(B.u, o); pv = ldo(B.v, o);
        if (t < 128) {
            const int nb = strip_block(t, n.nL, n.nR, n.nB, n.nT);
            const unsigned so = boff<T>(nb) + strip_pick(sk.kb, nb == n.ib);
            sh = ldo(B.h, so); sz = ldo(B.zb, so); su = ldo(B.u, so); sv = ldo(B.v, so);
        }
    };
    const int nwg = gridDim.x / NXCD, first = R.start + nwg;
    const bool more = R.end > first;
    int pos = R.start + blockIdx.x / NXCD;
    int g = 1;  // the next position to read
    Nb cur;
    if (pos < R.end) {
        cur = block_nb<BATCH>(P, pos);
        fetch(cur);
    }
    if (more) queue_take_now(qc, first, s.next, 1, t);
    for (int npos; pos < R.end; pos = npos) {
        Q4<T> qv;
        qv.a = ph; qv.b = DEV ? pz : pz + ph; qv.c = pu; qv.d = pv;
        s.q[tix(x, y)] = qv;
        {
            if (t < 128) {
                Q4<T> r;
                r.a = sh; r.b = DEV ? sz : sz + sh; r.c = su; r.d = sv;
                s.q[cs] = r;
            }
        }
        if (more) queue_take_now(qc, first, s.next, g + 1, t);
        __syncthreads();
        const Nb n = cur;
        npos = more ? queue_read(s.next, g++) : R.end;
        if (npos < R.end) {
            cur = block_nb<BATCH>(P, npos);
            fetch(cur);
        }
        if (BATCH) {
            if (n.sid != csid) {
                if (csid >= 0) wave_flush<T, FAST>(C, L + csid, smax, t);
                csid = n.sid;
                smax = T(0.0);
            }
            if (ldu(&L[n.sid].done, 0)) continue;
        }
        T dh, dhu, dhv;
        CellFaces<T> A;
        const bool w = blk_wall(P, n.ib, n.nL, n.nR, n.nB, n.nT);
        const T dtc = tile_fluxes<T, FAST, true>(s, C, t, qv, w && n.nL == n.ib, w && n.nR == n.ib, w && n.nB == n.ib,
                                                 w && n.nT == n.ib, A, dh, dhu, dhv);
        if (EXT && P.bopen && (n.nL == n.ib || n.nR == n.ib || n.nB == n.ib || n.nT == n.ib))
            // boundary values at the predictor's time, totaltime + dt/2 with the previous dt (src/FlowCPU.cu:94)
            open_sides<T, FAST>(A, qv, C, P, t, n.ib, n.nL, n.nR, n.nB, n.nT, L->totaltime + L->dt * 0.5, B.h, B.u, B.v,
                                B.zb, dh, dhu, dhv);
        if (EXT && P.nriver) dh = river_inflow<T>(P, n.ib, x, y, L->totaltime, dh);
        const unsigned oi = boff_i<T>(n.ib) + ki;
        stno(B.dh, oi, dh);
        stno(B.dhu, oi, dhu);
        stno(B.dhv, oi, dhv);
        smax = dmax(smax, dtc);
    }
    if (BATCH) {
        if (csid >= 0) wave_flush<T, FAST>(C, L + csid, smax, t);
        return;
    }
    const T m = -block_min(-smax, s.red, t);
    if (t == 0) slot_min(L, blockIdx.x, speed_dt<T, FAST>(C, m));
}

// Kahan step: h + d with the running compensation c (Kahan 1965).
template <class T> __device__ __forceinline__ T kahan_add(T h, T d, T& c) {
    const T y = d - c;
    const T t = h + y;
    c = (t - h) - y;
    return t;
}

// Persistent corrector with the same schedule and prefetch, through each XCD's
// range from its end: the predictor left the last blocks' lines in the caches
// (16.33 ms against 16.43 for ten steps at 8192 x 8192 cells).  COMP: the depth
// update accumulates with a compensated (Kahan) sum, so the small increments
// of rain and of slow flows are not lost to FP32 rounding of h.
template <class T, bool FAST, bool BATCH, bool COMP, bool EXT>
__device__ __forceinline__ void corrector_body(const KParams& P, const Cst<T>& C, const StepBuffers<T>& B, DevLoop* L,
                                               DevLoop* Lnext, int mode) {
    LoopState S;
    if (!BATCH) S = step_state<T>(L, Lnext, mode);
    if (blockIdx.x == 0 && threadIdx.x < NXCD) P.queue[threadIdx.x * QSTRIDE] = 0;  // the predictor's
    if (!BATCH && !S.go) return;
    __shared__ Tile<T, FAST> s;
    const int t = threadIdx.x;
    const int x = t & 15, y = t >> 4;
    const int xcd = blockIdx.x % NXCD;
    const Range R = xcd_range(xcd, P.nblk);
    int* const qc = P.queue + (NXCD + xcd) * QSTRIDE;
    const int cs = strip_cell(t);
    const StripK sk = strip_k<T>(t);
    const int fmc = P.ForceMassConserve;
    T ph = T(0), pu = T(0), pv = T(0), pdh = T(0), pdhu = T(0), pdhv = T(0), pz = T(0), pcf = T(0), pch = T(0);
    T sh = T(0), su = T(0), sv = T(0), sdh = T(0), sdhu = T(0), sdhv = T(0), sz = T(0);
    const unsigned kb = (unsigned)memloc(x, y, 0) * sizeof(T);
    const unsigned ki = (unsigned)(y * BW + x) * sizeof(T);  // in the tendency arrays
    auto fetch = [&](const Nb& n) {
        const int ib = n.ib;
        const unsigned o = boff<T>(ib) + kb, oi = boff_i<T>(ib) + ki;
        ph = ldo(B.h, o); pu = ldo(B.u, o); pv = ldo(B.v, o);
        pdh = ldo(B.dh, oi); pdhu = ldo(B.dhu, oi); pdhv = ldo(B.dhv, oi);
        pz = ldo(B.zb, o);
        if (COMP) pch = ldo(B.ch, oi);
        if (!(BATCH ? ldu(&L[n.sid].cf_uniform, 0) : P.cf_uniform)) pcf = ldno(B.cf, o);
        if (t < 128) {
            const int nb = strip_block(t, n.nL, n.nR, n.nB, n.nT);
            const bool self = nb == ib;
            const unsigned so = boff<T>(nb) + strip_pick(sk.kb, self);
            const unsigned soi = boff_i<T>(nb) + strip_pick(sk.ki, self);
            sh = ldo(B.h, so); su = ldo(B.u, so); sv = ldo(B.v, so);
            sdh = ldo(B.dh, soi); sdhu = ldo(B.dhu, soi); sdhv = ldo(B.dhv, soi);
            sz = ldo(B.zb, so);
        }
    };
    // The step's dt and rain rate are uniform over a launch (one domain).
    const T dt_one = BATCH ? T(0) : uniform(T(S.dt));
    const T rate_one = BATCH ? T(0) : uniform(sizeof(T) == 8 ? T(S.rate64) : T(S.rate32));
    const int nwg = gridDim.x / NXCD, first_pos = R.start + nwg;
    const bool more = R.end > first_pos;
    int pend = 0;
    if (more && t == 0) pend = queue_take(qc);
    int pos = R.start + blockIdx.x / NXCD;
    int g = 1;  // the next position to read
    Nb cur;
    if (pos < R.end) {
        cur = block_nb<BATCH>(P, R.start + R.end - 1 - pos);
        fetch(cur);
    }
    for (int npos; pos < R.end; pos = npos) {
        const DevLoop* Lm = L + (BATCH ? cur.sid : 0);
        if (BATCH && !ldu(&Lm->go, 0)) {
            if (more) queue_publish(qc, first_pos, s.next, g, t, pend);
            __syncthreads();
            npos = more ? queue_read(s.next, g++) : R.end;
            if (npos < R.end) {
                cur = block_nb<BATCH>(P, R.start + R.end - 1 - npos);
                fetch(cur);
            }
            continue;
        }
        const T dt = BATCH ? T(lds_f64(&Lm->dt)) : dt_one;
        const T hdt = dt * T(0.5);
        // this block's U^n (kept for the full-step advance) and its U* tile
        const bool cfu = BATCH ? ldu(&Lm->cf_uniform, 0) : P.cf_uniform;
        const T h0 = ph, u0 = pu, v0 = pv, zb0 = pz,
                cf0 = cfu ? T(BATCH ? lds_f64(&Lm->cf_value) : P.cf_value) : pcf;
        T comp = pch;
        // Consume the prefetched values here, where the loads are waited for
        // anyway, so that no wait inside the block's arithmetic can stall on
        // the next block's prefetch.
        asm volatile("" ::"v"(h0), "v"(u0), "v"(v0), "v"(zb0), "v"(cf0));
        if (COMP) asm volatile("" ::"v"(comp));
        Q4<T> qs;
        advance<T, FAST>(C, fmc, hdt, h0, u0, v0, pdh, pdhu, pdhv, qs.a, qs.c, qs.d);
        qs.b = FAST ? zb0 : zb0 + qs.a;
        s.q[tix(x, y)] = qs;
        {
            if (t < 128) {
                Q4<T> r;
                advance<T, FAST>(C, fmc, hdt, sh, su, sv, sdh, sdhu, sdhv, r.a, r.c, r.d);
                r.b = FAST ? sz : sz + r.a;
                s.q[cs] = r;
            }
        }
        if (more) queue_publish(qc, first_pos, s.next, g, t, pend);
        __syncthreads();
        const Nb n = cur;
        npos = more ? queue_read(s.next, g++) : R.end;
        if (npos < R.end) {
            cur = block_nb<BATCH>(P, R.start + R.end - 1 - npos);
            fetch(cur);
        }
        const int ib = n.ib, nL = n.nL, nR = n.nR, nB = n.nB, nT = n.nT;
        T dh, dhu, dhv;
        CellFaces<T> A;
        const bool w = blk_wall(P, ib, nL, nR, nB, nT);
        (void)tile_fluxes<T, FAST, false>(s, C, t, qs, w && nL == ib, w && nR == ib, w && nB == ib, w && nT == ib, A, dh,
                                          dhu, dhv);
        if (EXT && P.bopen && (nL == ib || nR == ib || nB == ib || nT == ib))
            // boundary values at totaltime + dt, from the step-start state (src/FlowCPU.cu:187)
            open_sides<T, FAST>(A, qs, C, P, t, ib, nL, nR, nB, nT, S.tcorr, B.h, B.u, B.v, B.zb, dh, dhu, dhv);
        if (EXT && P.nriver) dh = river_inflow<T>(P, ib, x, y, S.tstart, dh);
        T h1, u1, v1;
        const unsigned oc = boff<T>(ib) + kb, oci = boff_i<T>(ib) + ki;  // this block's cells
        if (COMP) {
            // advance() with the depth increment added through the compensated sum
            T m;
            const bool lim = dry_limit(C, fmc, dt, h0, dh, m);
            h1 = kahan_add(h0, lim ? -m : dt * dh, comp);
            const T r = Ar<T, FAST>::rcp(h1);
            u1 = h1 > C.eps ? fma(h0, u0, dt * dhu) * r : T(0.0);
            v1 = h1 > C.eps ? fma(h0, v0, dt * dhv) * r : T(0.0);
        } else {
            advance<T, FAST>(C, fmc, dt, h0, u0, v0, dh, dhu, dhv, h1, u1, v1);
        }
        // the implicit uniform rain after cleanup (src/Updateforcing.cu:530-581): its depth
        T rainhh = T(0.0);
        if (P.rain_on) {
            T act = (double)zb0 < C.mask_d ? T(1.0) : T(0.0);
            if (EXT) {
                rainhh = rain_depth<T>(P, S, ib, x, y, dt) * act;
            } else {
                const T rate = BATCH ? (sizeof(T) == 8 ? T(lds_f64(&Lm->rate64)) : T(lds_f32(&Lm->rate32))) : rate_one;
                const T a = rate * dt;
                rainhh = (a < T(0.0) ? T(0.0) : a) * act;  // std::max(a, 0)
            }
        }
        if (FAST) {
            // Bottom friction (src/Friction.cu:89-148) and the rain's dilution of the momentum in
            // one reciprocal: where h > eps, u and v scale by 1 / (1 + tb) for the friction and
            // then by h / (h + rain) for the rain (the rain's wetness test, (double)h > eps, is
            // the same as h > T(eps) for every float h), i.e. by h / ((1 + tb) (h + rain)).
            // Manning's tb = g n^2 dt |u| h^(-1/3) / h takes h^(-4/3) as one exp2(log2(h) (-4/3)).
            if (h1 > C.eps) {
                typedef Ar<T, FAST> A;
                const T normu = A::sqrt_(u1 * u1 + v1 * v1);
                T k;  // tb / |u|
                if (P.frictionmodel == 0) {
                    k = cf0 * dt * A::rcp(h1);
                } else if (P.frictionmodel == 1) {
                    T Hbar = h1 / cf0;
                    T cfi;
                    if (Hbar <= T(2.71828182845905)) cfi = T(1.0) / (T(0.46) * Hbar);
                    else cfi = T(1.0) / (T(2.5) * (log(Hbar) - T(1.0) + T(1.359) / Hbar));
                    k = cfi * cfi * dt * A::rcp(h1);
                } else {
                    k = (C.g * cf0 * cf0 * dt) * (T)exp2f(-1.33333337f * log2f((float)h1));
                }
                const T tb = k * normu;
                const T r = h1 * A::rcp(fma(tb, h1 + rainhh, h1 + rainhh));
                u1 = u1 * r;
                v1 = v1 * r;
            }
            h1 = COMP ? kahan_add(h1, rainhh, comp) : h1 + rainhh;
        } else {
            // bottom friction, src/Friction.cu:89-148
            if (h1 > C.eps) {
                T normu = sqrt(u1 * u1 + v1 * v1);
                T cfi;
                if (P.frictionmodel == 0) {
                    cfi = cf0;
                } else if (P.frictionmodel == 1) {
                    T Hbar = h1 / cf0;
                    if (Hbar <= T(2.71828182845905)) cfi = T(1.0) / (T(0.46) * Hbar);
                    else cfi = T(1.0) / (T(2.5) * (log(Hbar) - T(1.0) + T(1.359) / Hbar));
                    cfi = cfi * cfi;
                } else {
                    cfi = C.g * cf0 * cf0 / cbrt(h1);
                }
                T tb = cfi * normu / h1 * dt;
                u1 = u1 / (T(1.0) + tb);
                v1 = v1 / (T(1.0) + tb);
            }
            if (P.rain_on) {
                T qvol = h1 / (h1 + rainhh);
                bool wetold = (double)h1 > C.eps_d;
                h1 = h1 + rainhh;
                if (wetold) {
                    u1 = u1 * qvol;
                    v1 = v1 * qvol;
                }
            }
        }
        stno(B.ho, oc, h1);
        stno(B.uo, oc, u1);
        stno(B.vo, oc, v1);
        if (COMP) sto(B.ch, oci, comp);
        if (P.hmax) {
            const float hv = (float)h1;
            const unsigned of = boff<float>(ib) + (unsigned)memloc(x, y, 0) * 4u;
            if (hv > ldo(P.hmax, of)) sto(P.hmax, of, hv);
        }
    }
    queue_end(t, pend);
}

// Waves per SIMD asked of the plain one-level corrector: six for the FAST
// forms, which then hold to 80 VGPRs (84 unbounded, a sixth of the waves
// less); five for exact FP32, whose 93 VGPRs spill at six (1,118 us against
// 1,150 for ten rain steps on 1520 x 2032 cells); FP64 takes what its 160
// VGPRs allow.  Batches and the forcing kernels (open boundaries, rivers, rain
// maps) need more registers: they run as k_corrector_wide, the FP32 forcing
// ones held to four waves, the others unbounded (forced into 80 VGPRs the
// batch corrector measured 3 % slower).
template <class T, bool FAST, bool BATCH, bool COMP>
__global__ __launch_bounds__(256, sizeof(T) == 8 ? 3 : FAST ? 6 : 5) void k_corrector(KParams P, Cst<T> C, StepBuffers<T> B, DevLoop* L, DevLoop* Lnext, int mode) {
    static_assert(!BATCH, "batches use k_corrector_wide");
    corrector_body<T, FAST, false, COMP, false>(P, C, B, L, Lnext, mode);
}
template <class T, bool FAST, bool BATCH, bool COMP, bool EXT>
__global__ __launch_bounds__(256, EXT && sizeof(T) == 4 ? 4 : 1) void k_corrector_wide(KParams P, Cst<T> C, StepBuffers<T> B, DevLoop* L, DevLoop* Lnext, int mode) {
    corrector_body<T, FAST, BATCH, COMP, EXT>(P, C, B, L, Lnext, mode);
}

// One wave per loop state: reduce_dt_wave (the slots' minimum, clamp, landing, time keeping).
template <class T> __global__ __launch_bounds__(64) void k_reduce_dt(DevLoop* L, DevLoop* Lnext, int mode) {
    reduce_dt_wave<T>(L + blockIdx.x, Lnext + blockIdx.x, mode);
}

// Output statistics after a step (Calcmeanmax, src/Meanmax.cu:15-112), all
// in one pass over the state: with mask & 1 the sums of h, zs, u, v
// (addavg_var, :374-400), U = |(u, v)|, h U and h U U assigned as
// addUandhU does (:495-525), all seven divided by the step count at an
// output step, nextoutputtime - totaltime <= dt * T(1e-5) (divavg_var,
// :434-460); with mask & 2 the maxima of h, zs, u, v, U, h U, h (u^2 + v^2)
// (max_var, max_Norm, max_hU, max_hUU, :560-660); with mask & 4 the wet time
// (addwettime, :786-818).  zs is zb + h.  IEEE square roots and divisions in
// every precision.
template <class T>
__global__ __launch_bounds__(256) void k_stats(KParams P, StatsLaunch S, const T* __restrict__ hh,
                                               const T* __restrict__ uu, const T* __restrict__ vv,
                                               const T* __restrict__ zb, const DevLoop* L, int advanced) {
    if (!L->go) return;
    const int ib = P.active[blockIdx.x];
    const int i = memloc(threadIdx.x & 15, threadIdx.x >> 4, ib);
    const T h = hh[i], u = uu[i], v = vv[i], zs = zb[i] + h;
    if (S.mask & 1) {
        const double tt = advanced ? L->totaltime : L->totaltime + L->dt;
        const bool divide = L->nextoutputtime - tt <= L->dt * (double)T(0.00001);
        const T n = T(L->stats_n);
        const T U = sqrt((u * u) + (v * v));
        const T m[7] = {((T*)S.a[0])[i] + h, ((T*)S.a[1])[i] + zs, ((T*)S.a[2])[i] + u, ((T*)S.a[3])[i] + v,
                        U, h * U, h * U * U};
#pragma unroll
        for (int k = 0; k < 7; k++) ((T*)S.a[k])[i] = divide ? m[k] / n : m[k];
    }
    if (S.mask & 2) {
        const T U = sqrt((u * u) + (v * v));
        const T x[7] = {h, zs, u, v, U, h * U, h * (u * u + v * v)};
#pragma unroll
        for (int k = 0; k < 7; k++) {
            T* const p = (T*)S.a[7 + k];
            const T o = p[i];
            p[i] = o < x[k] ? x[k] : o;
        }
    }
    if ((S.mask & 4) && h > T(S.wet_threshold)) ((T*)S.a[14])[i] = ((T*)S.a[14])[i] + T(L->dt);
}

template <class T> __global__ __launch_bounds__(256) void k_stats_reset(KParams P, StatsLaunch S, int which) {
    const int ib = P.active[blockIdx.x];
    const int i = memloc(threadIdx.x & 15, threadIdx.x >> 4, ib);
    const T neg = -std::numeric_limits<T>::max();  // Loop.hugenegval (src/Mainloop.cu:233-234)
#pragma unroll
    for (int k = 0; k < 15; k++) {
        const int bit = k < 7 ? 1 : k < 14 ? 2 : 4;
        if ((which & bit) && (S.mask & bit)) ((T*)S.a[k])[i] = (k >= 7 && k < 14) ? neg : T(0);
    }
}

void launch_stats(int precision, const KParams& P, const StatsLaunch& S, const void* h, const void* u, const void* v,
                  const void* zb, const DevLoop* L, int advanced, hipStream_t st) {
    if (!S.mask || P.nblk <= 0) return;
    if (precision == 0)
        hipLaunchKernelGGL(k_stats<double>, dim3(P.nblk), dim3(256), 0, st, P, S, (const double*)h, (const double*)u,
                           (const double*)v, (const double*)zb, L, advanced);
    else
        hipLaunchKernelGGL(k_stats<float>, dim3(P.nblk), dim3(256), 0, st, P, S, (const float*)h, (const float*)u,
                           (const float*)v, (const float*)zb, L, advanced);
}

void launch_stats_reset(int precision, const KParams& P, const StatsLaunch& S, int which, hipStream_t st) {
    if (!S.mask || P.nblk <= 0) return;
    if (precision == 0) hipLaunchKernelGGL(k_stats_reset<double>, dim3(P.nblk), dim3(256), 0, st, P, S, which);
    else hipLaunchKernelGGL(k_stats_reset<float>, dim3(P.nblk), dim3(256), 0, st, P, S, which);
}

// The rain map of a step, at its start: InterpstepCPU (src/GridManip.cu:602-622)
// between the frames that bracket totaltime (Forcingthisstep,
// src/Updateforcing.cu:61-127), in double, stored as float.
__global__ __launch_bounds__(256) void k_rain_now(KParams P, const DevLoop* L) {
    const int n = P.rnx * P.rny;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n || L->done) return;
    const double tt = L->totaltime;
    const int k = min(max((int)floor((tt - P.rt0) / P.rdtf), 0), P.rnframes - 2);
    const float uo = P.rframes[(size_t)k * n + i], un = P.rframes[(size_t)(k + 1) * n + i];
    P.rnow[i] = (float)((double)uo + (tt - P.rdtf * k) * (double)(un - uo) / P.rdtf);
}

// Level maps of the boundary segments at the step's start (Forcingthisstep on
// each segment's WLmap, src/Updateforcing.cu:29-35, 83-126): InterpstepCPU
// (src/GridManip.cu:602-622) between the frames bracketing totaltime, with its
// hdstep*hddt that omits the first frame's time.  One row of workgroups per segment.
__global__ __launch_bounds__(256) void k_bnd_now(KParams P, const DevLoop* L) {
    const BSeg& S = P.seg[blockIdx.y];
    const int n = S.nx * S.ny;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (!S.frames || i >= n || L->done) return;
    const double tt = L->totaltime;
    const int k = min(max((int)floor((tt - S.to) / S.tdt), 0), S.nt - 2);
    const float uo = S.frames[(size_t)k * n + i], un = S.frames[(size_t)(k + 1) * n + i];
    S.now[i] = (float)((double)uo + (tt - S.tdt * k) * (double)(un - uo) / S.tdt);
}

void launch_rain_now(const KParams& P, const DevLoop* L, hipStream_t st) {
    if (P.bmapmax > 0)
        hipLaunchKernelGGL(k_bnd_now, dim3((P.bmapmax + 255) / 256, P.nseg), dim3(256), 0, st, P, L);
    if (!P.rframes || P.rnframes < 2) return;
    hipLaunchKernelGGL(k_rain_now, dim3((P.rnx * P.rny + 255) / 256), dim3(256), 0, st, P, L);
}

// Per-cell initial step delta/sqrt(g*max(h,eps)) and its block minimum,
// src/Mainloop.cu:569-589.
template <class T>
__global__ __launch_bounds__(256) void k_init_dt(KParams P, const T* __restrict__ h, DevLoop* L) {
    __shared__ T red[4];
    const int t = threadIdx.x;
    const int ib = P.active[blockIdx.x];
    const int i = memloc(t & 15, t >> 4, ib);
    T d = calcres(T(P.delta0), P.level[ib]) / sqrt(T(P.g) * (h[i] > T(P.eps) ? h[i] : T(P.eps)));
    T m = block_min(d, red, t);
    if (t == 0) slot_min(L + (P.sid ? P.sid[ib] : 0), blockIdx.x, m);
}

// Running maximum depth of the interior cells (output path of src/Meanmax.cu:15-120).
template <class T>
__global__ __launch_bounds__(256) void k_maxdepth(KParams P, const T* __restrict__ h, float* __restrict__ hmax) {
    const int t = threadIdx.x;
    const int i = memloc(t & 15, t >> 4, P.active[blockIdx.x]);
    const float v = (float)h[i];
    if (v > hmax[i]) hmax[i] = v;
}

template <class T> __global__ void k_gauges(const T* __restrict__ h, const int* __restrict__ cell, float* val, int n) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) val[k] = cell[k] >= 0 ? (float)h[cell[k]] : __builtin_nanf("");
}

template <class T>
__global__ void k_gauge_step(const T* __restrict__ h, const int* __restrict__ cell, const DevLoop* L, int n, int cap,
                             float* ring, double* tring) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int m = k >> 4;
    const DevLoop& Lm = L[m];
    if (!Lm.go || Lm.gevery <= 0 || Lm.nstep % Lm.gevery != 0) return;
    const int s = Lm.nstep / Lm.gevery - 1;
    if (s >= cap) return;
    if (cell[k] >= 0) ring[(size_t)k * cap + s] = (float)h[cell[k]];
    if ((k & 15) == 0) tring[(size_t)m * cap + s] = Lm.totaltime;
}

template <class T>
__global__ __launch_bounds__(256) void k_refine_flags(KParams P, const T* __restrict__ a, const T* __restrict__ b,
                                                      int mode, T lo, T hi, unsigned char* flags) {
    const int t = threadIdx.x;
    const int ib = P.active[blockIdx.x];
    const int x = t & 15, y = t >> 4;
    const int i = memloc(x, y, ib);
    auto val = [&](int c) { return b ? b[c] + a[c] : a[c]; };
    const T z = val(i);
    int hit;
    if (mode == 0) hit = z > lo;
    else if (mode == 1) hit = z >= lo && z <= hi;
    else {
        // steepness: a difference to the next interior cell over the cell size
        const T d = T(calcres(P.delta0, P.level[ib]));
        const T gx = x < BW - 1 ? fabs(val(memloc(x + 1, y, ib)) - z) / d : T(0);
        const T gy = y < BW - 1 ? fabs(val(memloc(x, y + 1, ib)) - z) / d : T(0);
        hit = gx > lo || gy > lo;
    }
    const int any = __syncthreads_or(hit);
    if (t == 0) flags[ib] = any ? 1 : 0;
}

// Block partial sums of h*delta^2 in FP64 (deterministic two-level sum).
template <class T>
__global__ __launch_bounds__(256) void k_volume(KParams P, const T* __restrict__ h, double* __restrict__ part) {
    __shared__ double red[4];
    const int t = threadIdx.x;
    const int ib = P.active[blockIdx.x];
    const double d = calcres(P.delta0, P.level[ib]);
    double v = (double)h[memloc(t & 15, t >> 4, ib)] * d * d;
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((t & 63) == 0) red[t >> 6] = v;
    __syncthreads();
    if (t == 0) part[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

__global__ __launch_bounds__(1024) void k_sum(const double* __restrict__ part, int n, double* out) {
    __shared__ double red[16];
    const int t = threadIdx.x;
    double v = 0.0;
    for (int k = t; k < n; k += 1024) v += part[k];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((t & 63) == 0) red[t >> 6] = v;
    __syncthreads();
    if (t == 0) {
        double s2 = 0.0;
        for (int k = 0; k < 16; k++) s2 += red[k];
        *out = s2;
    }
}

// The loop state enters a run in the arguments of a launch and leaves it in
// host memory that the last launch writes (out, may be null), both in stream
// order: with a copy and a wait at either end, and a third wait for the settled
// state, a step called by itself took 64 us on 256 x 256 cells in FP64.
__global__ __launch_bounds__(64) void k_set_loop(LoopState S, DevLoop* L) {
    slots_empty(L);
    if (threadIdx.x == 0) *(LoopState*)L = S;
}
static_assert(sizeof(LoopState) % 4 == 0 && sizeof(LoopState) <= 256, "a lane copies a word");
__device__ __forceinline__ void loop_out(const DevLoop* L, LoopState* out) {
    if (out && blockIdx.x == 0 && threadIdx.x < sizeof(LoopState) / 4)
        ((int*)out)[threadIdx.x] = ((const int*)(const LoopState*)L)[threadIdx.x];
}
__global__ __launch_bounds__(64) void k_loop_out(const DevLoop* L, LoopState* out) { loop_out(L, out); }

// cleanupGPU semantics (src/Advection.cu:399-417): copy interior h, u, v of
// the blocks whose state ended in the second buffer (odd step count).
template <class T>
__global__ __launch_bounds__(256) void k_settle(KParams P, const T* __restrict__ h, const T* __restrict__ u,
                                                const T* __restrict__ v, T* __restrict__ ho, T* __restrict__ uo,
                                                T* __restrict__ vo, const DevLoop* L, LoopState* out) {
    const int t = threadIdx.x;
    loop_out(L, out);
    const int ib = P.active[blockIdx.x];
    if (!(L[P.sid ? P.sid[ib] : 0].steps_done & 1)) return;
    const int i = memloc(t & 15, t >> 4, ib);
    ho[i] = h[i];
    uo[i] = u[i];
    vo[i] = v[i];
}

// The caller's device state for a step on its own arrays (bgf_step_device):
// k_import copies the interior cells of h, u, v of the active blocks into the
// handle's state; k_export writes the step's result back into the caller's
// h, zs = zb + h (what the next step recomputes, src/Halo.cu:72-107), u, v and,
// when keep is set, into the handle's step-start buffer as well.
template <class T>
__global__ __launch_bounds__(256) void k_import(KParams P, const T* __restrict__ h, const T* __restrict__ u,
                                                const T* __restrict__ v, T* __restrict__ hd, T* __restrict__ ud,
                                                T* __restrict__ vd) {
    const int i = memloc(threadIdx.x & 15, threadIdx.x >> 4, P.active[blockIdx.x]);
    hd[i] = h[i];
    ud[i] = u[i];
    vd[i] = v[i];
}
template <class T>
__global__ __launch_bounds__(256) void k_export(KParams P, const T* __restrict__ h, const T* __restrict__ u,
                                                const T* __restrict__ v, const T* __restrict__ zb, T* __restrict__ ho,
                                                T* __restrict__ zso, T* __restrict__ uo, T* __restrict__ vo,
                                                T* __restrict__ hk, T* __restrict__ uk, T* __restrict__ vk,
                                                const DevLoop* L, LoopState* out) {
    loop_out(L, out);
    const int i = memloc(threadIdx.x & 15, threadIdx.x >> 4, P.active[blockIdx.x]);
    const T hh = h[i], uu = u[i], vv = v[i];
    ho[i] = hh;
    zso[i] = zb[i] + hh;
    uo[i] = uu;
    vo[i] = vv;
    if (hk) {
        hk[i] = hh;
        uk[i] = uu;
        vk[i] = vv;
    }
}

// ------------------------------------------------------------------ launch
// Workgroups of kernel k resident at once on the device (CUs x occupancy at
// 256 threads), a multiple of NXCD; 0 if the query fails.
template <class K> int resident_wgs(K kernel) {
    int dev = 0, ncu = 0, occ = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, 256, 0) != hipSuccess) return 0;
    return ncu * (occ < 1 ? 1 : occ) / NXCD * NXCD;
}
// A persistent launch's grid: the schedule's count, held to what the kernel
// that is actually launched keeps resident (the forcing and batch variants
// need more registers than the plain kernels the schedule was sized for).
inline int fit_grid(int grid, int resident) {
    return resident >= NXCD && grid > resident ? resident : grid;
}

template <class T, bool FAST, bool BATCH, bool COMP>
void launch_step_t(const KParams& P, const StepBuffers<T>& B, DevLoop* L, DevLoop* Lnext, int advance_time,
                   hipStream_t st, hipEvent_t* ev) {
    if (!BATCH) launch_rain_now(P, L, st);
    if (ev) (void)hipEventRecord(ev[0], st);
    const Cst<T> C = make_cst<T, FAST>(P);
    // batches never take the extra forcings: only one-level handles get the EXT kernels
    constexpr bool EXT_OK = !BATCH;
    const bool ext = EXT_OK && (P.bopen || P.nriver || P.rnow);
    static const int res_pred = resident_wgs(k_predictor<T, FAST, BATCH, FAST>);
    static const int res_pred_ext = resident_wgs(k_predictor<T, FAST, BATCH, FAST, EXT_OK>);
    static const int res_corr = BATCH ? resident_wgs(k_corrector_wide<T, FAST, true, COMP, false>)
                                      : resident_wgs(k_corrector<T, FAST, false, COMP>);
    static const int res_corr_ext = resident_wgs(k_corrector_wide<T, FAST, false, COMP, true>);
    const int gp = fit_grid(P.grid_pred, ext ? res_pred_ext : res_pred);
    const int gc = fit_grid(P.grid_corr, ext ? res_corr_ext : res_corr);
    if (ext) hipLaunchKernelGGL((k_predictor<T, FAST, BATCH, FAST, EXT_OK>), dim3(gp), dim3(256), 0, st, P, C, B, L);
    else hipLaunchKernelGGL((k_predictor<T, FAST, BATCH, FAST>), dim3(gp), dim3(256), 0, st, P, C, B, L);
    if (ev) (void)hipEventRecord(ev[1], st);
    if (BATCH) hipLaunchKernelGGL((k_reduce_dt<T>), dim3(P.nmember), dim3(64), 0, st, L, L, advance_time);
    if (ev) (void)hipEventRecord(ev[2], st);
    if constexpr (BATCH)
        hipLaunchKernelGGL((k_corrector_wide<T, FAST, true, COMP, false>), dim3(gc), dim3(256), 0, st, P, C, B, L, Lnext,
                           advance_time);
    else if (ext)
        hipLaunchKernelGGL((k_corrector_wide<T, FAST, false, COMP, true>), dim3(gc), dim3(256), 0, st, P, C, B, L, Lnext,
                           advance_time);
    else
        hipLaunchKernelGGL((k_corrector<T, FAST, false, COMP>), dim3(gc), dim3(256), 0, st, P, C, B, L, Lnext,
                           advance_time);
    if (ev) (void)hipEventRecord(ev[3], st);
}

template <class T, bool FAST, bool COMP>
void launch_step_b(const KParams& P, const void* buffers, DevLoop* L, DevLoop* Lnext, int advance_time, hipStream_t st,
                   hipEvent_t* ev) {
    const StepBuffers<T>& B = *(const StepBuffers<T>*)buffers;
    if (P.sid) launch_step_t<T, FAST, true, COMP>(P, B, L, Lnext, advance_time, st, ev);
    else launch_step_t<T, FAST, false, COMP>(P, B, L, Lnext, advance_time, st, ev);
}

void launch_step(int precision, const KParams& P, const void* buffers, DevLoop* L, DevLoop* Lnext, int advance_time,
                 hipStream_t st, hipEvent_t* ev) {
    if (precision == 0) launch_step_b<double, false, false>(P, buffers, L, Lnext, advance_time, st, ev);
    else if (precision == 1) launch_step_b<float, false, false>(P, buffers, L, Lnext, advance_time, st, ev);
    else if (precision == 2) launch_step_b<float, true, false>(P, buffers, L, Lnext, advance_time, st, ev);
    else launch_step_b<float, true, true>(P, buffers, L, Lnext, advance_time, st, ev);
}

// Persistent grid: all workgroups resident at once (CUs x occupancy), a
// multiple of NXCD, and no more than the blocks need.  most: workgroups per CU
// that a grid not asked for by wg_per_cu takes at the most.  The FP32
// predictors fit seven by their registers, but the seventh starts late (its
// first block waits for another workgroup's end, and the launch for it) and
// more of them only lengthen the tail.  A step on rain, exact FP32, with seven,
// six, five and four, us: 720 x 640 cells 41.4, 33.8, 34.2, 34.6; 1024 x 1024
// 56.0, 50.4, 49.4, 49.3; 1520 x 1520 87.2, 80.4, 81.6, 83.9; 2048 x 2048 134,
// 128.5, 131, 137; 4096 x 4096 478.6, 476.6, 487.4, 499; 8192 x 8192 1896,
// 1899, 1943, 2002: six, within 0.2 % of the best from 1520 x 1520 on and 2 %
// below.  FAST, seven, six, five, four: 33.0, 26.2, 25.6, 25.6; 45.2, 38.7,
// 37.9, 37.4; 68.6, 63.2, 62.0, 61.7; 105.2, 102.2, 101.2, 100.9; 375, 374,
// 372, 375; 1475, 1473, 1472, 1500: five, within 1.3 %.  Smaller grids have
// fewer blocks than that.
template <class K> int grid_for(K kernel, int nblk, int wg_per_cu, int most = 8) {
    int dev = 0, ncu = 0, occ = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, 256, 0) != hipSuccess) return 0;
    occ = std::min(occ, wg_per_cu > 0 ? wg_per_cu : most);
    if (occ < 1) occ = 1;
    long nwg = (long)ncu * occ;
    long need = ((long)nblk + NXCD - 1) / NXCD * NXCD;
    if (nwg > need) nwg = need;
    nwg = (nwg + NXCD - 1) / NXCD * NXCD;
    return (int)nwg;
}

int persistent_grid(int precision, int corrector, int nblk, int wg_per_cu) {
    const int w = wg_per_cu;
    if (precision == 0)
        return corrector ? grid_for(k_corrector<double, false, false, false>, nblk, w)
                         : grid_for(k_predictor<double, false, false, false>, nblk, w);
    if (precision == 1)
        return corrector ? grid_for(k_corrector<float, false, false, false>, nblk, w)
                         : grid_for(k_predictor<float, false, false, false>, nblk, w, 6);
    if (precision == 2)
        return corrector ? grid_for(k_corrector<float, true, false, false>, nblk, w)
                         : grid_for(k_predictor<float, true, false, true>, nblk, w, 5);
    return corrector ? grid_for(k_corrector<float, true, false, true>, nblk, w)
                     : grid_for(k_predictor<float, true, false, true>, nblk, w, 5);
}

void launch_init_dt(int precision, const KParams& P, const void* h, DevLoop* L, hipStream_t st) {
    if (precision == 0) {
        hipLaunchKernelGGL(k_init_dt<double>, dim3(P.nblk), dim3(256), 0, st, P, (const double*)h, L);
        hipLaunchKernelGGL(k_reduce_dt<double>, dim3(P.sid ? P.nmember : 1), dim3(64), 0, st, L, L, 2);
    } else {
        hipLaunchKernelGGL(k_init_dt<float>, dim3(P.nblk), dim3(256), 0, st, P, (const float*)h, L);
        hipLaunchKernelGGL(k_reduce_dt<float>, dim3(P.sid ? P.nmember : 1), dim3(64), 0, st, L, L, 2);
    }
}

void launch_init_dt_member(int precision, const KParams& P, const void* h, DevLoop* L, int member, hipStream_t st) {
    if (precision == 0) {
        hipLaunchKernelGGL(k_init_dt<double>, dim3(P.nblk), dim3(256), 0, st, P, (const double*)h, L);
        hipLaunchKernelGGL(k_reduce_dt<double>, dim3(1), dim3(64), 0, st, L + member, L + member, 2);
    } else {
        hipLaunchKernelGGL(k_init_dt<float>, dim3(P.nblk), dim3(256), 0, st, P, (const float*)h, L);
        hipLaunchKernelGGL(k_reduce_dt<float>, dim3(1), dim3(64), 0, st, L + member, L + member, 2);
    }
}

void launch_maxdepth(int precision, const KParams& P, const void* h, float* hmax, hipStream_t st) {
    if (precision == 0) hipLaunchKernelGGL(k_maxdepth<double>, dim3(P.nblk), dim3(256), 0, st, P, (const double*)h, hmax);
    else hipLaunchKernelGGL(k_maxdepth<float>, dim3(P.nblk), dim3(256), 0, st, P, (const float*)h, hmax);
}

void launch_gauges(int precision, const void* h, const int* cell, float* val, int n, hipStream_t st) {
    const dim3 g((n + 255) / 256), b(256);
    if (precision == 0) hipLaunchKernelGGL(k_gauges<double>, g, b, 0, st, (const double*)h, cell, val, n);
    else hipLaunchKernelGGL(k_gauges<float>, g, b, 0, st, (const float*)h, cell, val, n);
}

void launch_gauge_step(int precision, const void* h, const int* cell, const DevLoop* L, int nmember, int cap,
                       float* ring, double* tring, hipStream_t st) {
    const int n = 16 * nmember;
    const dim3 g((n + 255) / 256), b(256);
    if (precision == 0) hipLaunchKernelGGL(k_gauge_step<double>, g, b, 0, st, (const double*)h, cell, L, n, cap, ring, tring);
    else hipLaunchKernelGGL(k_gauge_step<float>, g, b, 0, st, (const float*)h, cell, L, n, cap, ring, tring);
}

void launch_refine_flags(int precision, const KParams& P, const void* a, const void* b, int mode, double lo,
                         double hi, unsigned char* flags, hipStream_t st) {
    if (precision == 0)
        hipLaunchKernelGGL(k_refine_flags<double>, dim3(P.nblk), dim3(256), 0, st, P, (const double*)a,
                           (const double*)b, mode, lo, hi, flags);
    else
        hipLaunchKernelGGL(k_refine_flags<float>, dim3(P.nblk), dim3(256), 0, st, P, (const float*)a,
                           (const float*)b, mode, (float)lo, (float)hi, flags);
}

void launch_reduce_dt(int precision, DevLoop* L, DevLoop* Lnext, int nloop, int advance_time, hipStream_t st) {
    if (precision == 0)
        hipLaunchKernelGGL(k_reduce_dt<double>, dim3(nloop), dim3(64), 0, st, L, Lnext, advance_time);
    else hipLaunchKernelGGL(k_reduce_dt<float>, dim3(nloop), dim3(64), 0, st, L, Lnext, advance_time);
}

void launch_volume(int precision, const KParams& P, const void* h, double* part, double* out, hipStream_t st) {
    if (precision == 0) hipLaunchKernelGGL(k_volume<double>, dim3(P.nblk), dim3(256), 0, st, P, (const double*)h, part);
    else hipLaunchKernelGGL(k_volume<float>, dim3(P.nblk), dim3(256), 0, st, P, (const float*)h, part);
    hipLaunchKernelGGL(k_sum, dim3(1), dim3(1024), 0, st, part, P.nblk, out);
}

void launch_set_loop(const LoopState& S, DevLoop* L, hipStream_t st) {
    hipLaunchKernelGGL(k_set_loop, dim3(1), dim3(64), 0, st, S, L);
}

void launch_loop_out(const DevLoop* L, LoopState* out, hipStream_t st) {
    hipLaunchKernelGGL(k_loop_out, dim3(1), dim3(64), 0, st, L, out);
}

void launch_settle(int precision, const KParams& P, const void* const* src, void* const* dst, const DevLoop* L,
                   LoopState* out, hipStream_t st) {
    if (precision == 0)
        hipLaunchKernelGGL(k_settle<double>, dim3(P.nblk), dim3(256), 0, st, P, (const double*)src[0],
                           (const double*)src[1], (const double*)src[2], (double*)dst[0], (double*)dst[1],
                           (double*)dst[2], L, out);
    else
        hipLaunchKernelGGL(k_settle<float>, dim3(P.nblk), dim3(256), 0, st, P, (const float*)src[0],
                           (const float*)src[1], (const float*)src[2], (float*)dst[0], (float*)dst[1],
                           (float*)dst[2], L, out);
}

void launch_import(int precision, const KParams& P, const void* const* src, void* const* dst, hipStream_t st) {
    if (P.nblk <= 0) return;
    if (precision == 0)
        hipLaunchKernelGGL(k_import<double>, dim3(P.nblk), dim3(256), 0, st, P, (const double*)src[0],
                           (const double*)src[1], (const double*)src[2], (double*)dst[0], (double*)dst[1],
                           (double*)dst[2]);
    else
        hipLaunchKernelGGL(k_import<float>, dim3(P.nblk), dim3(256), 0, st, P, (const float*)src[0],
                           (const float*)src[1], (const float*)src[2], (float*)dst[0], (float*)dst[1],
                           (float*)dst[2]);
}

void launch_export(int precision, const KParams& P, const void* const* src, const void* zb, void* const* dst,
                   void* const* keep, const DevLoop* L, LoopState* lout, hipStream_t st) {
    if (P.nblk <= 0) return;
    if (precision == 0)
        hipLaunchKernelGGL(k_export<double>, dim3(P.nblk), dim3(256), 0, st, P, (const double*)src[0],
                           (const double*)src[1], (const double*)src[2], (const double*)zb, (double*)dst[0],
                           (double*)dst[1], (double*)dst[2], (double*)dst[3], keep ? (double*)keep[0] : nullptr,
                           keep ? (double*)keep[1] : nullptr, keep ? (double*)keep[2] : nullptr, L, lout);
    else
        hipLaunchKernelGGL(k_export<float>, dim3(P.nblk), dim3(256), 0, st, P, (const float*)src[0],
                           (const float*)src[1], (const float*)src[2], (const float*)zb, (float*)dst[0],
                           (float*)dst[1], (float*)dst[2], (float*)dst[3], keep ? (float*)keep[0] : nullptr,
                           keep ? (float*)keep[1] : nullptr, keep ? (float*)keep[2] : nullptr, L, lout);
}

// Interior cells of n blocks, field by field of each (zs = zb + h, h, u, v
// where asked), BSI values apiece, to host memory that the GPU can reach.
template <class T>
__global__ __launch_bounds__(256) void k_pack_state(const int* active, const T* zb, const T* h, const T* u, const T* v,
                                                    int fields, T* out) {
    const int t = threadIdx.x, c = memloc(t & 15, t >> 4, ldu(active, blockIdx.x));
    T* o = out + (size_t)blockIdx.x * __builtin_popcount(fields) * BSI + t;
    if (fields & 1) { *o = zb[c] + h[c]; o += BSI; }
    if (fields & 2) { *o = h[c]; o += BSI; }
    if (fields & 4) { *o = u[c]; o += BSI; }
    if (fields & 8) *o = v[c];
}

void launch_pack_state(int precision, const int* active, int n, const void* zb, const void* h, const void* u,
                       const void* v, int fields, void* out, hipStream_t st) {
    if (precision == 0)
        hipLaunchKernelGGL(k_pack_state<double>, dim3(n), dim3(256), 0, st, active, (const double*)zb, (const double*)h,
                           (const double*)u, (const double*)v, fields, (double*)out);
    else
        hipLaunchKernelGGL(k_pack_state<float>, dim3(n), dim3(256), 0, st, active, (const float*)zb, (const float*)h,
                           (const float*)u, (const float*)v, fields, (float*)out);
}

}  // namespace bgf
