// bgf_common.h -- device helpers shared by the one-level kernels
// (bgf_kernels.hip) and the multi-level kernels (bgf_amr.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <limits>

#include "bgf_arith.h"
#include "bgf_kernels.h"

namespace bgf {

constexpr int BW = 16;      // cells per block side (src/Param.h:52)
constexpr int MW = 18;      // stored tile side: one halo cell each way
constexpr int BS = MW * MW; // values per block
constexpr int BSI = BW * BW; // values per block of the interior-only tendency arrays

// src/MemManagement.cu:37-40
__device__ __forceinline__ int memloc(int i, int j, int ib) { return (i + 1) + (j + 1) * MW + ib * BS; }

// LDS pitches.  128-bit accesses of 16-lane rows are free of bank conflicts
// on gfx950 only at pitches of 16 or 32 entries (17 to 24 cost 4 conflict
// cycles per read, measured with SQ_LDS_BANK_CONFLICT), so the arrays that are
// only read by rows (y slopes, Y faces) are 16 wide; the others, which also
// take column accesses (halo strips, the ring, the 17th faces), keep odd
// pitches.
constexpr int TP = 21;  // tile: x, y in [-2, 17]
constexpr int GXP = 19; // x slopes: x in [-1, 16], y in [0, 15]
constexpr int GYP = 16; // y slopes: x in [0, 15], y in [-1, 16]
constexpr int FP = 17;  // X faces xf in [0, 16], y in [0, 15]

__device__ __forceinline__ int tix(int x, int y) { return (y + 2) * TP + (x + 2); }
__device__ __forceinline__ int gxi(int x, int y) { return y * GXP + (x + 1); }
__device__ __forceinline__ int gyi(int x, int y) { return (y + 1) * GYP + x; }

// fmin/fmax (v_min/v_max, fused into v_min3/v_max3).  They differ from the
// reference's std::min/std::max only for NaN operands and in the sign of a
// zero result, neither of which changes any value of the step.
__device__ __forceinline__ float dmax(float a, float b) { return fmaxf(a, b); }
__device__ __forceinline__ float dmin(float a, float b) { return fminf(a, b); }
__device__ __forceinline__ double dmax(double a, double b) { return fmax(a, b); }
__device__ __forceinline__ double dmin(double a, double b) { return fmin(a, b); }

// A cell's (h, zs, u, v), a cell's four gradients, or a face's four fluxes.
template <class T> struct alignas(4 * sizeof(T)) Q4 {
    T a, b, c, d;
};

// Holds the end of a face's arithmetic in front of the next face's: the
// compiler otherwise sinks it past the barrier to the stores, and the operands
// of three faces outgrow the registers that the occupancy allows (83 VGPRs in
// FP32 and 163 in FP64 against 60 and 110).
template <class T> __device__ __forceinline__ void finish(Q4<T>& F) {
    asm volatile("" : "+v"(F.a), "+v"(F.b), "+v"(F.c), "+v"(F.d)::"memory");
}

// Block indices are workgroup-uniform: read them through the constant address
// space so they become scalar loads, which do not wait behind the vector
// loads of the prefetch.
__device__ __forceinline__ int ldu(const int* p, int i) {
    return ((const __attribute__((address_space(4))) int*)p)[i];
}
__device__ __forceinline__ double lds_f64(const double* p) {
    return *(const __attribute__((address_space(4))) double*)p;
}
__device__ __forceinline__ float lds_f32(const float* p) {
    return *(const __attribute__((address_space(4))) float*)p;
}
// The contiguous range of n positions that XCD xcd takes: workgroup b of a
// launch of n workgroups runs on XCD b % NXCD and is the (b / NXCD)-th there.
struct Range {
    int start, end;
};
__device__ __forceinline__ Range xcd_range(int xcd, int n) {
    const int per = n / NXCD, rem = n % NXCD;
    Range R;
    R.start = xcd * per + (xcd < rem ? xcd : rem);
    R.end = R.start + per + (xcd < rem ? 1 : 0);
    return R;
}

// Division and square root: IEEE in EXACT kernels, hardware approximations in FAST ones.
template <class T, bool FAST> struct Ar {
    __device__ static __forceinline__ T rcp(T a) { return T(1.0) / a; }
    __device__ static __forceinline__ T sqrt_(T a) { return sqrt(a); }
};
template <> struct Ar<float, true> {
    __device__ static __forceinline__ float rcp(float a) { return __builtin_amdgcn_rcpf(a); }
    __device__ static __forceinline__ float sqrt_(float a) { return __builtin_amdgcn_sqrtf(a); }
};

// The four quotients of a Q4.
template <class T> __device__ __forceinline__ Q4<T> div4(const FixedDiv<T>& K, const Q4<T>& x) {
    Q4<T> q{quick_div(K, x.a), quick_div(K, x.b), quick_div(K, x.c), quick_div(K, x.d)};
    if (__builtin_expect(odd_div(K, x.a) | odd_div(K, x.b) | odd_div(K, x.c) | odd_div(K, x.d), 0))
        q = Q4<T>{x.a / K.d, x.b / K.d, x.c / K.d, x.d / K.d};
    return q;
}

// 1 / b rounded as IEEE division rounds it (rounded_rcp), from the hardware's
// reciprocal.
__device__ __forceinline__ double plain_rcp(double b) { return rounded_rcp(b, __builtin_amdgcn_rcp(b)); }
__device__ __forceinline__ float plain_rcp(float b) { return rounded_rcp(b, __builtin_amdgcn_rcpf(b)); }

// The step that the drying limiter allows (src/Advection.cu:349-352):
// min(dt, max(h, eps) / |dh|) evaluated in double, where dh < 0.  The limiter
// binds only where max(h, eps) < dt |dh|; a product a few roundings larger
// decides that for nearly every cell, and only the others divide.  epsT: eps
// rounded to T, which may differ from eps in its last bit.
template <class T> __device__ __forceinline__ T dry_step(T dt, T h, T dh, T epsT, double eps) {
    T edt = dt;
    if (!(dh >= T(0.0)) && !(dmax(h, epsT) > dt * -dh * T(1.0 + 0x1p-18))) {
        const double m = (double)h < eps ? eps : (double)h;
        const double lim = m / (double)fabs(dh);
        edt = T(lim < (double)dt ? lim : (double)dt);
    }
    return edt;
}

// Workgroup minimum over 256 threads (four wave64s); every thread gets it.
template <class T> __device__ __forceinline__ T block_min(T v, T* red, int t) {
    for (int off = 32; off > 0; off >>= 1) {
        T o = __shfl_xor(v, off, 64);
        v = o < v ? o : v;
    }
    if ((t & 63) == 0) red[t >> 6] = v;
    __syncthreads();
    T m = red[0];
#pragma unroll
    for (int k = 1; k < 4; k++) m = red[k] < m ? red[k] : m;
    return m;
}

// Positive floating-point values order like their bit patterns, so a block
// minimum merges into a dt slot with an integer atomic min.
__device__ __forceinline__ void slot_min(DevLoop* L, int k, float v) {
    atomicMin(&L->slot32[k & (NSLOT - 1)], __float_as_uint(v));
}
__device__ __forceinline__ void slot_min(DevLoop* L, int k, double v) {
    atomicMin(&L->slot64[k & (NSLOT - 1)], (unsigned long long)__double_as_longlong(v));
}

// Minimum of a loop state's slots, by a whole wave.
template <class T> __device__ __forceinline__ T slots_min(const DevLoop* L) {
    const int l = threadIdx.x & 63;
    T m = sizeof(T) == 8 ? (T)__longlong_as_double((long long)L->slot64[l]) : (T)__uint_as_float(L->slot32[l]);
    for (int off = 32; off > 0; off >>= 1) {
        const T o = __shfl_xor(m, off, 64);
        m = o < m ? o : m;
    }
    return m;
}
__device__ __forceinline__ void slots_empty(DevLoop* L) {
    const int l = threadIdx.x & 63;
    L->slot32[l] = 0x7f800000u;
    L->slot64[l] = 0x7ff0000000000000ull;
}

// The first entry k from lo on of a series of increasing times t with
// t[k] > tt (or >= tt where AT), or its last entry n - 1.  By halves: the
// entries are read one after the other, and a series by the minute over days
// has thousands.
template <bool AT> __device__ __forceinline__ int series_entry(const double* t, int lo, int n, double tt) {
    int hi = n - 1;
    while (lo < hi) {
        const int m = (lo + hi) >> 1;
        const double d = t[m] - tt;
        if (AT ? d < 0.0 : d <= 0.0) lo = m + 1;
        else hi = m;
    }
    return lo;
}

// A loop state past the dt reduction of its step, from the slots' minimum m:
// the smaller of m and 1/epsi, the clamp and the output-time landing of
// CalctimestepCPU in FP64.  mode 0: a step that leaves totaltime to the caller;
// 1: a step followed by totaltime += dt; 2: the initial dt only.
template <class T> __device__ __forceinline__ void advance_loop(LoopState& L, T m, int mode) {
    if (L.done) {
        L.go = 0;
        return;
    }
    const T epsi = sizeof(T) == 8 ? T(2.220446049250313e-16) : T(1.1920928955078125e-07);
    if (L.rain_n > 0) {
        // the uniform rain of this step, at its start (Forcingthisstep,
        // src/Updateforcing.cu:45-60, interptime src/Util_CPU.cu:107-110)
        const double tt = L.totaltime;
        const int k = series_entry<true>(L.rain_t, 1, L.rain_n, tt);
        const double prev = L.rain_v[k - 1];
        const double now = prev + (tt - L.rain_t[k - 1]) / (L.rain_t[k] - L.rain_t[k - 1]) * (L.rain_v[k] - prev);
        L.rain = now;
        L.rate64 = now / 1000.0 / 3600.0;
        L.rate32 = (float)now / 1000.0f / 3600.0f;
    }
    L.tstart = L.totaltime;
    L.tpred = L.totaltime + L.dt * 0.5;
    T dt = T(1.0) / epsi;
    dt = m < dt ? m : dt;
    if ((double)dt > 1.5 * L.dtmax) dt = T(1.5 * L.dtmax);
    double rem = L.nextoutputtime - L.totaltime;
    if (ceil(rem / (double)dt) > 0.0) dt = T(rem / ceil(rem / (double)dt));
    L.dt = (double)dt;
    L.dtmax = (double)dt;
    L.tcorr = L.totaltime + L.dt;
    if (!isfinite((double)dt) || dt <= T(0)) L.bad |= 1;
    if (mode != 2) {
        L.go = 1;
        L.steps_done = L.steps_done + 1;
        L.nstep = L.nstep + 1;
        L.stats_n = L.stats_n + 1;
    }
    if (mode == 1) {
        L.totaltime = L.totaltime + L.dt;
        if (L.totaltime >= L.endtime) L.done = 1;
        // CrashDetection (src/Mainloop.cu:648-660): after the step that advanced the time
        if (L.dt < L.dtmin && L.totaltime < L.endtime) {
            L.crashed = 1;
            L.done = 1;
        }
    }
}

// The reduction as a launch of its own, one wave per loop state: L's state past
// it goes to Lnext (L itself for batches), with empty slots.
template <class T> __device__ __forceinline__ void reduce_dt_wave(const DevLoop* L, DevLoop* Lnext, int mode) {
    LoopState S = *L;
    advance_loop<T>(S, slots_min<T>(L), mode);
    slots_empty(Lnext);
    if (threadIdx.x == 0) *(LoopState*)Lnext = S;
}

// The state of a step past its dt reduction, worked out by every wave of the
// launch that follows the predictor from the predictor's state L; the first
// wave of workgroup 0 leaves it in Lnext.  A reduction launch of its own took
// 4.7 us a step, a third of what a small domain's other two launches need.
template <class T> __device__ __forceinline__ LoopState step_state(const DevLoop* L, DevLoop* Lnext, int mode) {
    LoopState S = *L;
    advance_loop<T>(S, slots_min<T>(L), mode);
    if (blockIdx.x == 0 && threadIdx.x < 64) {
        if (threadIdx.x == 0) *(LoopState*)Lnext = S;
        slots_empty(Lnext);
    }
    return S;
}

// calcres (src/Util_CPU.cu:194-198): cell size of a level.
template <class T> __device__ __forceinline__ T calcres(T dx, int level) {
    return level < 0 ? dx * T(1 << -level) : dx / T(1 << level);
}

// Rain rate [mm/h] of the current rain map at cell (ix, iy) of block ib, as
// AddrainforcingImplicitCPU samples it (src/Updateforcing.cu:549-558): the
// cell position in T, then interp2BUQ (src/GridManip.cu:520-560) in double.
template <class T> __device__ __forceinline__ T rain_map_rate(const KParams& P, int ib, int ix, int iy) {
    const T delta = calcres(T(P.dx), P.level[ib]);
    const T x = T(P.xo) + T(P.bxo[ib]) + T(ix) * delta;
    const T y = T(P.yo) + T(P.byo[ib]) + T(iy) * delta;
    const double xmax = P.rxo + (P.rnx - 1) * P.rdx, ymax = P.ryo + (P.rny - 1) * P.rdx;
    const double xi = fmax(fmin((double)x, xmax), P.rxo);
    const double yi = fmax(fmin((double)y, ymax), P.ryo);
    int cfi = (int)floor((xi - P.rxo) / P.rdx);
    cfi = min(max(cfi, 0), P.rnx - 2);
    int cfj = (int)floor((yi - P.ryo) / P.rdx);
    cfj = min(max(cfj, 0), P.rny - 2);
    const int cfip = cfi + 1, cfjp = cfj + 1;
    const double x1 = P.rxo + P.rdx * cfi, x2 = P.rxo + P.rdx * cfip;
    const double y1 = P.ryo + P.rdx * cfj, y2 = P.ryo + P.rdx * cfjp;
    const double q11 = P.rnow[cfi + cfj * P.rnx], q12 = P.rnow[cfi + cfjp * P.rnx];
    const double q21 = P.rnow[cfip + cfj * P.rnx], q22 = P.rnow[cfip + cfjp * P.rnx];
    // BilinearInterpolation (src/Util_CPU.cu:129-144)
    const double x2x1 = x2 - x1, y2y1 = y2 - y1, x2x = x2 - xi, y2y = y2 - yi, yy1 = yi - y1, xx1 = xi - x1;
    return T(1.0 / (x2x1 * y2y1) * (q11 * x2x * y2y + q21 * xx1 * y2y + q12 * x2x * yy1 + q22 * xx1 * yy1));
}

// The per-step rain depth of a cell, m: max(rate / 1000 / 3600 * dt, 0)
// (src/Updateforcing.cu:560) from the rain map, or from the loop's uniform
// rate (precomputed as rate64 / rate32).
template <class T>
__device__ __forceinline__ T rain_depth(const KParams& P, const LoopState& L, int ib, int ix, int iy, T dt) {
    T a;
    if (P.rnow) a = rain_map_rate<T>(P, ib, ix, iy) / T(1000.0) / T(3600.0) * dt;
    else a = (sizeof(T) == 8 ? T(L.rate64) : T(L.rate32)) * dt;
    return a < T(0.0) ? T(0.0) : a;  // std::max(a, 0)
}

// ------------------------------------------------------ boundary types 2, 3
// The boundary type of block ib's boundary faces: its segment's, or aoibnd
// without segments.
__device__ __forceinline__ int blk_btype(const KParams& P, int ib) {
    return P.bseg ? P.seg[P.bseg[ib]].type : P.aoibnd;
}

// Whether block ib's boundary faces (if it has any) are walls.
__device__ __forceinline__ bool blk_wall(const KParams& P, int ib, int nL, int nR, int nB, int nT) {
    return (nL == ib || nR == ib || nB == ib || nT == ib) && blk_btype(P, ib) == 0;
}

// The water level a boundary face of segment S takes at stage time t, as the
// float zsbnd of bndFluxGPUSideCPU plus Param.zsoffset (src/Boundary.cu:587-648):
// the segment's uniform series at t (FlowbndFlux, src/Boundary.cu:116-145: the
// bracketing entries, interptime); or its level map of this step sampled at
// the face, (XParam.xo + xx, XParam.yo + yy) with xx = XBlock.xo + ix*delta
// formed in T and ix = 0 or 16 across the block (interp2BUQ,
// src/GridManip.cu:531-574, in double); or, without forcing, zs0.
template <class T>
__device__ __forceinline__ float seg_level(const KParams& P, const BSeg& S, double t, int ib, int ix, int iy) {
    float z;
    if (S.now) {
        const T delta = calcres(T(P.dx), P.level[ib]);
        const double x = P.xo + (double)(T(P.bxo[ib]) + T(ix) * delta);
        const double y = P.yo + (double)(T(P.byo[ib]) + T(iy) * delta);
        const double xmax = S.xo + (S.nx - 1) * S.dx, ymax = S.yo + (S.ny - 1) * S.dy;
        const double xi = fmax(fmin(x, xmax), S.xo);
        const double yi = fmax(fmin(y, ymax), S.yo);
        const int cfi = min(max((int)floor((xi - S.xo) / S.dx), 0), S.nx - 2);
        const int cfj = min(max((int)floor((yi - S.yo) / S.dy), 0), S.ny - 2);
        const int cfip = cfi + 1, cfjp = cfj + 1;
        const double x1 = S.xo + S.dx * cfi, x2 = S.xo + S.dx * cfip;
        const double y1 = S.yo + S.dy * cfj, y2 = S.yo + S.dy * cfjp;
        const double q11 = S.now[cfi + cfj * S.nx], q12 = S.now[cfi + cfjp * S.nx];
        const double q21 = S.now[cfip + cfj * S.nx], q22 = S.now[cfip + cfjp * S.nx];
        // BilinearInterpolation (src/Util_CPU.cu:129-144)
        const double x2x1 = x2 - x1, y2y1 = y2 - y1, x2x = x2 - xi, y2y = y2 - yi, yy1 = yi - y1, xx1 = xi - x1;
        z = (float)(1.0 / (x2x1 * y2y1) * (q11 * x2x * y2y + q21 * xx1 * y2y + q12 * x2x * yy1 + q22 * xx1 * yy1));
    } else if (S.on) {
        const int k = series_entry<true>(S.t, 1, S.n, t);  // the reference does not stop at the end
        z = (float)(S.z[k - 1] + (t - S.t[k - 1]) / (S.t[k] - S.t[k - 1]) * (S.z[k] - S.z[k - 1]));
    } else {
        z = (float)S.zs0;
    }
    return (float)((double)z + P.bzsoffset);  // zsbnd = zsbnd + zsoffset (src/Boundary.cu:648)
}

// The boundary taper at stage time t (FlowbndFlux, src/Boundary.cu:124-128): a
// segment with forcing ramps its level in over Param.bndtaper seconds from
// Param.inittime.
template <class T> __device__ __forceinline__ T bnd_taper(const KParams& P, const BSeg& S, double t) {
    return S.on && P.btaper > 0.0 ? T(fmin((t - P.binittime) / P.btaper, 1.0)) : T(1.0);
}

// Mass flux through a boundary face of type 2 (Dirichlet1Q) or 3 (ABS1DQ)
// from the step-start state at the face cell (zsi, hi) and the inside cell
// (zsin, hin, and its normal velocity unin), bndFluxGPUSideCPU
// (src/Boundary.cu:587-741, 1943-2032) with the face's level zsbnd (offset
// included) and the taper, without atmospheric pressure, and with the
// absorbing boundary's qmean filter at rest (it moves only with a fixed
// Param.dt, and stays 0 otherwise).  Returns false
// where the reference falls back to the no-slip patch (a dry face that the
// boundary level does not flood).
template <class T>
__device__ __forceinline__ bool bnd_flux(const KParams& P, int s, int type, float zsbnd, T taper, T zsi, T hi, T zsin,
                                         T hin, T unin, T& q) {
    const T sign = (s == 1 || s == 3) ? T(1.0) : T(-1.0);
    const T zsatm = T(0.0);
    const T zsX = T(((double)(T(zsbnd) + zsatm) - 0.5 * (double)(zsi + zsin)) * (double)taper +
                    0.5 * (double)(zsi + zsin));
    if (!((double)hi > P.eps || zsX > zsi)) return false;
    const T g = T(P.g);
    if (type == 3) {
        const T qmean = hi < T(0.01) ? T(0.0) : T(0.0) * q + T(1.0) * (T(1.0) - T(0.0)) * T(0.0);
        const T zn = zsX < zsi - hi ? zsi - hi : zsX;
        const T hn = hi < T(0.0001) ? T(0.0001) : hi;
        const T un = sign * sqrt(g / hn) * (zsi - zn);
        q = un * hn + qmean;
    } else {
        const T zbin = zsin - hin;
        const T a = hin < T(0.0) ? T(0.0) : hin;
        const T b = zsX - zbin < T(0.0) ? T(0.0) : zsX - zbin;
        const T un = sign * T(2.0) * (sqrt(g * a) - sqrt(g * b)) + unin;
        q = un * hin;
    }
    return true;
}

// ------------------------------------------------------------------ rivers
// Discharges added to the depth tendency of cell (ix, iy) of block ib, river
// by river (InjectRiverCPU, src/Updateforcing.cu:314-363): a cell receives a
// river's rate when its box, formed in T, overlaps the river's (OBBdetect,
// src/Util_CPU.cu:286-296); only blocks that held a discharge cell when the
// rivers were set (or the mesh last changed) are visited.  The rate is the
// flow at tt, the step's start, over the discharge area (AddRiverForcing,
// src/Updateforcing.cu:146-165): interpolated between the first entry later
// than tt and the one before, where it is used (a launch of its own for it
// took 4.6 us a step).
template <class T>
__device__ __forceinline__ T river_inflow(const KParams& P, int ib, int ix, int iy, double tt, T dh) {
    // Few blocks hold discharge cells: laid out for the others.  Without the hint the FP64 corrector stage of
    // the multi-level step came out 450 instructions longer (9.56 ms for ten steps of 39,348 blocks, now 9.41).
    if (__builtin_expect(!P.nriver || !P.rblk[ib], 1)) return dh;
    const T levdx = calcres(T(P.dx), P.level[ib]);
    const T xllo = T(P.xo + P.bxo[ib]), yllo = T(P.yo + P.byo[ib]);
    const T xl = xllo + T(ix) * levdx - T(0.5) * levdx, yb = yllo + T(iy) * levdx - T(0.5) * levdx;
    const T xr = xllo + T(ix) * levdx + T(0.5) * levdx, yt = yllo + T(iy) * levdx + T(0.5) * levdx;
    for (int r = 0; r < P.nriver; r++) {
        const double* b = P.rbox + 4 * r;
        const bool tx = T(b[0]) <= xr && T(b[1]) >= xl;
        const bool ty = T(b[2]) <= yt && T(b[3]) >= yb;
        if (tx && ty) {
            const double* t = P.rt + P.roff[r];
            const double* q = P.rq + P.roff[r];
            const int n = P.roff[r + 1] - P.roff[r];
            const int e = series_entry<false>(t, 0, n, tt);  // the reference does not stop at the end
            const int a = e - 1 > 0 ? e - 1 : 0;
            const double flow = q[a] + (tt - t[a]) / (t[e] - t[a]) * (q[e] - q[a]);
            // the reference's array of rates is a T
            dh += sizeof(T) == 8 ? T(flow / P.rarea[r]) : T((double)(float)flow / P.rarea[r]);
        }
    }
    return dh;
}

}  // namespace bgf
