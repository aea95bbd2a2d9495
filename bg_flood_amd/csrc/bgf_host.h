// bgf_host.h -- host-side helpers shared by the C ABI translation units:
// error reporting, parameter checks and the processing order of the
// persistent kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <limits>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/bgflood_amd.h"
#include "bgf_kernels.h"

namespace bgf_host {

constexpr int BW = 16;
constexpr int MW = 18;
constexpr int BS = MW * MW;
constexpr int BSI = BW * BW;  // values per block of the interior-only arrays (tendencies, compensation)

inline thread_local std::string g_err;

inline bgf_status fail(bgf_status s, const std::string& msg) {
    g_err = msg;
    return s;
}

#define HIPCHK(call)                                                                                   \
    do {                                                                                               \
        hipError_t e_ = (call);                                                                        \
        if (e_ != hipSuccess) return fail(BGF_ERR_HIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

inline int memloc(int i, int j, int ib) { return (i + 1) + (j + 1) * MW + ib * BS; }

// Whether a kernel may dereference p: device, managed or pinned host memory.  Pageable host
// memory (the usual mistake when device arrays are expected) makes the query fail; the error is
// cleared so it does not surface at the next HIP call.
inline bool device_accessible(const void* p) {
    if (!p) return false;
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type == hipMemoryTypeDevice || a.type == hipMemoryTypeManaged || a.type == hipMemoryTypeHost ||
           a.type == hipMemoryTypeUnified;
}

// Reading a state back: a kernel writes the interior cells of some blocks, and
// the sum zb + h, straight into pinned host memory, and the host spreads their
// rows over the caller's arrays (whose other cells stay as they are); one piece
// is written while the one before is spread, so the pinned memory stays small.
// Copying whole arrays, with their halos and the bed, through pageable memory
// took 3.48 ms for the eight members (25.6 MB of arrays) of an ensemble.  The
// pieces are no larger than the largest read through them needs, and one that
// suffices has no second: a domain of one block takes 8 KB, not 2 MB.
struct ReadBack {
    static constexpr size_t PIECE = 1024 * 1024;  // bytes of one of the two pieces at the most, a power of two
    unsigned char* mem[2] = {nullptr, nullptr};
    size_t size[2] = {0, 0};
    hipEvent_t ev[2] = {nullptr, nullptr};
    std::mutex busy;  // several threads may read the states of one batch
    ~ReadBack() {
        for (int k = 0; k < 2; k++) {
            if (ev[k]) (void)hipEventDestroy(ev[k]);
            if (mem[k]) (void)hipHostFree(mem[k]);
        }
    }
};

// Fields dst = (zs, h, u, v; null: not wanted) of the blocks active (d_active:
// the same list on the device), block ib going to place ib - off of dst.
// most: the blocks of the largest such read to expect (the members of a batch
// are read in turn).
inline bgf_status read_back(ReadBack& R, int prec, const std::vector<int>& active, int most, int off,
                            const int* d_active, const void* zb, const void* h, const void* u, const void* v,
                            void* const dst[4], hipStream_t st) {
    const size_t es = prec == 0 ? sizeof(double) : sizeof(float);
    int fields = 0, nf = 0;
    for (int k = 0; k < 4; k++)
        if (dst[k]) fields |= 1 << k, nf++;
    const int n = (int)active.size();
    if (!nf || !n) return BGF_OK;
    std::lock_guard<std::mutex> lock(R.busy);
    // the stream's device, which need not be the calling thread's current one
    struct OnDevice {
        int was = -1, dev = -1;
        ~OnDevice() { if (was >= 0 && was != dev) (void)hipSetDevice(was); }
    } on;
    HIPCHK(hipStreamGetDevice(st, &on.dev));
    HIPCHK(hipGetDevice(&on.was));
    if (on.was != on.dev) HIPCHK(hipSetDevice(on.dev));
    const int per = (int)(ReadBack::PIECE / (nf * BSI * es)), pieces = (n + per - 1) / per;
    auto fetch = [&](int k) -> hipError_t {
        const int b0 = k * per;
        bgf::launch_pack_state(prec, d_active + b0, std::min(per, n - b0), zb, h, u, v, fields, R.mem[k & 1], st);
        const hipError_t e = hipGetLastError();
        return e == hipSuccess ? hipEventRecord(R.ev[k & 1], st) : e;
    };
    for (int k = 0; k < (most > per ? 2 : 1); k++) {
        if (!R.ev[k]) HIPCHK(hipEventCreateWithFlags(&R.ev[k], hipEventDisableTiming));
        size_t need = 4096;  // doubled: at most eight times for a handle
        while (need < (size_t)std::min(per, most) * nf * BSI * es) need *= 2;
        if (R.size[k] >= need) continue;
        if (R.mem[k]) (void)hipHostFree(R.mem[k]);
        R.mem[k] = nullptr;
        R.size[k] = 0;
        void* p = nullptr;
        if (hipHostMalloc(&p, need, hipHostMallocDefault) != hipSuccess) {
            (void)hipGetLastError();
            return fail(BGF_ERR_OOM, "host allocation failed");
        }
        R.mem[k] = (unsigned char*)p;
        R.size[k] = need;
    }
    HIPCHK(fetch(0));
    for (int k = 0; k < pieces; k++) {
        if (k + 1 < pieces) HIPCHK(fetch(k + 1));
        HIPCHK(hipEventSynchronize(R.ev[k & 1]));
        const unsigned char* src = R.mem[k & 1];
        for (int b = k * per; b < std::min(n, (k + 1) * per); b++)
            for (int f = 0; f < 4; f++) {
                if (!dst[f]) continue;
                unsigned char* d = (unsigned char*)dst[f] + (size_t)memloc(0, 0, active[b] - off) * es;
                for (int j = 0; j < BW; j++, src += BW * es, d += MW * es) {
                    if (es == 4) std::memcpy(d, src, BW * 4);
                    else std::memcpy(d, src, BW * 8);
                }
            }
    }
    return BGF_OK;
}

// Room for the gather recipes and the list of fix-up blocks of a multi-level
// batch of cap block slots, in one allocation.
inline bool mesh_tables(size_t cap, int4** rcell, int2** rmeta, int** fix) {
    const size_t n = bgf::RECIPES * cap;
    if (hipMalloc((void**)rcell, n * (sizeof(int4) + sizeof(int2)) + cap * sizeof(int)) != hipSuccess) return false;
    *rmeta = (int2*)(*rcell + n);
    *fix = (int*)(*rmeta + n);
    return true;
}

inline double level_dx(double dx, int lev) { return lev < 0 ? dx * (1 << -lev) : dx / (1 << lev); }

constexpr double kPi = 3.14159265;  // src/General.h:6

// src/Spherical.cu:15-30 in T, with the reference's mixed precision: y is
// formed in double ((iy+0.5) is a double) and the last division is by the
// double 2*dphi.
template <class T> inline T calc_cm(T Radius, T delta, T yo, int iy) {
    T y = yo + (iy + 0.5) * delta / Radius * T(180.0 / kPi);
    T phi = y * T(kPi / 180.0);
    T dphi = delta / (T(2.0 * Radius));
    return T((std::sin(phi + dphi) - std::sin(phi - dphi)) / (2.0 * dphi));
}

// src/Spherical.cu:43-64 in T.
template <class T> inline T calc_fm(T Radius, T delta, T yo, T iy) {
    T dy = delta / Radius * T(180.0 / kPi);
    T y = yo + iy * dy;
    T phi = y * T(kPi / 180.0);
    return std::cos(phi);
}

// Great-circle distance by the haversine formula (src/Spherical.cu:70-87) and
// the area of a dx x dx (degrees) cell centred at (lon, lat): the mean of its
// lower and upper edge lengths times its meridional edge length
// (src/Spherical.cu:101-120), in double as the rivers' set-up evaluates it
// (src/InitialConditions.cu:385-388).
inline double haversin_d(double Radius, double lon1, double lat1, double lon2, double lat2) {
    const double r = kPi / 180.0;
    const double dphi = (lat2 - lat1) * r, dlbda = (lon2 - lon1) * r;
    const double sp = std::sin(dphi / 2.0), sl = std::sin(dlbda / 2.0);
    const double a = sp * sp + std::cos(lat1 * r) * std::cos(lat2 * r) * sl * sl;
    return Radius * (2.0 * std::atan2(std::sqrt(a), std::sqrt(1.0 - a)));
}
inline double cell_area_sphere(double Radius, double lon, double lat, double dx) {
    const double lon1 = lon - 0.5 * dx, lon2 = lon + 0.5 * dx, lat1 = lat - 0.5 * dx, lat2 = lat + 0.5 * dx;
    const double lower = haversin_d(Radius, lon1, lat1, lon2, lat1);
    const double upper = haversin_d(Radius, lon1, lat2, lon2, lat2);
    const double side = haversin_d(Radius, lon1, lat1, lon1, lat2);
    return 0.5 * (lower * side + upper * side);
}

template <class T> inline T calcres_t(T dx, int lev) { return lev < 0 ? dx * (1 << -lev) : dx / (1 << lev); }

// Metric terms of every block of a spherical grid, in the layout of
// bgf::MET_*: the X and Y Kurganov faces (src/Kurganov.cu:474-641,
// 1404-1565) and the tendencies (src/Advection.cu:160-254).  Computed on the
// host with the same libm as the reference CPU step.
template <class T>
inline std::vector<T> metric_table(const bgf_param* p, const bgf_blocks* b, int nblkmem) {
    std::vector<T> M((size_t)nblkmem * bgf::METRIC_STRIDE, T(0));
    for (int ibl = 0; ibl < p->nblk; ibl++) {
        const int ib = b->active[ibl];
        const int lev = b->level[ib];
        const T delta = calcres_t(T(p->delta), lev);
        const T yblk = T(b->yo[ib]);
        const T ybo_k = T(p->yo + (double)yblk);  // Kurganov: T(XParam.yo + XBlock.yo[ib])
        const T ybo_e = (T)p->yo + yblk;          // updateEV: (T)XParam.yo + XBlock.yo[ib]
        const T R = T(p->Radius);
        T* m = M.data() + (size_t)ib * bgf::METRIC_STRIDE;
        for (int iy = 0; iy < BW; iy++) m[bgf::MET_CMX + iy] = calc_cm(R, delta, ybo_k, iy);
        for (int iy = 0; iy <= BW; iy++) {
            m[bgf::MET_CMY + iy] = calc_cm(R, delta, ybo_k, iy);
            m[bgf::MET_FMY + iy] = calc_fm(R, delta, ybo_k, T(iy));
        }
        const int top = b->TopLeft[ib], bot = b->BotLeft[ib];
        for (int iy = 0; iy < BW; iy++) {
            T yup = T(iy) + T(1.0), ydwn = T(iy);
            if (iy == BW - 1 && b->level[top] > lev) yup = iy + T(0.75);
            if (iy == 0 && b->level[bot] > lev) ydwn = iy - T(0.25);
            m[bgf::MET_CME + iy] = calc_cm(R, delta, ybo_e, iy);
            m[bgf::MET_FMV + iy] = calc_fm(R, delta, ybo_e, ydwn);
            m[bgf::MET_FMVP + iy] = calc_fm(R, delta, ybo_e, yup);
            m[bgf::MET_FC + iy] = T(std::sin((ybo_e + calcres_t(T(p->dx), lev) * iy) * kPi / 180.0) * kPi / T(21600.0));
        }
    }
    return M;
}

// Cell indices are 32-bit ints, as memloc's (src/MemManagement.cu:37-40):
// at most this many allocated blocks (1.7e9 cells).
constexpr int kMaxBlocks = 2147483647 / BS;

// Block slots an array may hold so that every byte offset (block and cell) fits 32 bits: the fused
// kernels address their arrays as base + a 32-bit offset.
inline long long max_blocks_for(int precision) {
    const long long es = precision == 0 ? 8 : 4;
    return 4294967295LL / (BS * es);
}
inline bool block_bytes_ok(long long nblkmem, int precision) { return nblkmem <= max_blocks_for(precision); }

inline bgf_status check_param(const bgf_param* p) {
    if (!p) return fail(BGF_ERR_INVALID_ARG, "null param");
    if (p->engine != 2) return fail(BGF_ERR_UNSUPPORTED, "only engine 2 (Kurganov) is provided");
    if (p->spherical && !(p->Radius > 0.0)) return fail(BGF_ERR_INVALID_ARG, "spherical grids need Radius > 0");
    if (p->nblk <= 0 || p->nblkmem < p->nblk) return fail(BGF_ERR_INVALID_ARG, "need 0 < nblk <= nblkmem");
    if (!block_bytes_ok(p->nblkmem, p->precision))
        return fail(BGF_ERR_UNSUPPORTED, "nblkmem " + std::to_string(p->nblkmem) +
                                             ": the fused kernels address an array with 32-bit byte offsets (at most " +
                                             std::to_string(max_blocks_for(p->precision)) + " blocks at this precision)");
    if (p->nblkmem > kMaxBlocks)
        return fail(BGF_ERR_UNSUPPORTED, "nblkmem above " + std::to_string(kMaxBlocks) +
                                             " blocks: cell indices would not fit in 32 bits");
    if (p->precision < 0 || p->precision > 3) return fail(BGF_ERR_INVALID_ARG, "bad precision");
    if (p->aoibnd != 0 && p->aoibnd != 1)
        return fail(BGF_ERR_UNSUPPORTED, "remainder boundary type must be 0 (wall) or 1 (Neumann)");
    if (p->frictionmodel < -1 || p->frictionmodel > 1) return fail(BGF_ERR_INVALID_ARG, "bad frictionmodel");
    if (!(p->delta > 0.0) || !(p->g > 0.0) || !(p->eps > 0.0)) return fail(BGF_ERR_INVALID_ARG, "bad g/eps/delta");
    return BGF_OK;
}

template <class T> inline double coriolis(double lat) {
    // src/Advection.cu:187 (Cartesian): sin(T(lat*pi/180))*pi/T(21600) with pi = 3.14159265
    const double pi = 3.14159265;
    return (double)T(std::sin(T(lat * pi / 180.0)) * pi / T(21600.0));
}

// Integer block coordinates of the active blocks (position among the blocks
// of their level), in active-list order.
struct BlockXY {
    std::vector<int> id;
    std::vector<long long> bx, by;
};
inline BlockXY block_xy(const bgf_blocks* b, int nblk, double dx) {
    BlockXY xy;
    xy.id.assign(b->active, b->active + nblk);
    xy.bx.resize(nblk);
    xy.by.resize(nblk);
    for (int k = 0; k < nblk; k++) {
        const int ib = b->active[k];
        const int lev = b->level[ib];
        const double levdx = lev < 0 ? dx * (1 << -lev) : dx / (1 << lev);
        xy.bx[k] = (long long)std::floor(b->xo[ib] / (BW * levdx));
        xy.by[k] = (long long)std::floor(b->yo[ib] / (BW * levdx));
    }
    return xy;
}

// Processing order of the persistent kernels: the active blocks grouped in
// tiles of tile_x x tile_y blocks (row-major tiles, row-major blocks inside a
// tile), by their integer block coordinates.  Each XCD processes consecutive
// positions of this order, so the blocks it has in flight at once form a
// compact patch whose neighbours are mostly in its own L2.  The tile is part
// of the launch schedule (bgf_set_schedule); TILE_X x TILE_Y is the default.
constexpr int TILE_X = 16, TILE_Y = 12;
inline std::vector<int> processing_order(const BlockXY& xy, int tile_x = TILE_X, int tile_y = TILE_Y) {
    const int nblk = (int)xy.id.size();
    long long maxbx = 1;
    for (int k = 0; k < nblk; k++)
        if (xy.bx[k] + 1 > maxbx) maxbx = xy.bx[k] + 1;
    const long long ntx = (maxbx + tile_x - 1) / tile_x;
    std::vector<long long> key(nblk);
    for (int k = 0; k < nblk; k++) {
        const long long tx = xy.bx[k] / tile_x, ty = xy.by[k] / tile_y;
        key[k] = ((ty * ntx + tx) * tile_y + xy.by[k] % tile_y) * tile_x + xy.bx[k] % tile_x;
    }
    std::vector<int> idx(nblk);
    for (int k = 0; k < nblk; k++) idx[k] = k;
    std::stable_sort(idx.begin(), idx.end(), [&](int a, int c) { return key[a] < key[c]; });
    std::vector<int> order(nblk);
    for (int k = 0; k < nblk; k++) order[k] = xy.id[idx[k]];
    return order;
}

// Neighbours of quadtree blocks from their integer positions: block k of the
// list has id[k], level lev[k] and position (ix[k], iy[k]) among the blocks
// of its level; the domain is nbx x nby blocks of level `base`.  A side shared
// with one block of the same or a coarser level points both halves at it, a
// side shared with two finer blocks points the first half (bottom or left)
// and the second half at them, a side on the domain edge points at the block
// itself (the convention of src/Mesh.cu:351-433 and src/Adaptation.cu:1017-1795).
// Outputs are indexed by block id.  Fails unless the blocks tile the domain
// with neighbouring levels within one of each other.
inline bgf_status quadtree_neighbours(int n, const int* id, const int* lev, const long long* ix, const long long* iy,
                                      int nbx, int nby, int base, int* LeftBot, int* LeftTop, int* RightBot,
                                      int* RightTop, int* TopLeft, int* TopRight, int* BotLeft, int* BotRight) {
    auto key = [base](int l, long long x, long long y) {
        return ((unsigned long long)(l - base) << 58) | ((unsigned long long)x << 29) | (unsigned long long)y;
    };
    int maxd = 0;
    for (int k = 0; k < n; k++) {
        const int d = lev[k] - base;
        if (d < 0 || d > 28) return fail(BGF_ERR_INVALID_ARG, "block level out of range");
        maxd = std::max(maxd, d);
    }
    // block positions: one dense grid per level while the finest grid is small (a few
    // million block positions), else a hash map
    std::vector<long long> off(maxd + 2, 0);
    for (int d = 0; d <= maxd; d++) off[d + 1] = off[d] + ((long long)nbx << d) * ((long long)nby << d);
    const bool dense = off[maxd + 1] <= (1LL << 24);
    std::vector<int> grid(dense ? (size_t)off[maxd + 1] : 0, -1);
    std::unordered_map<unsigned long long, int> at;
    if (!dense) at.reserve((size_t)n * 2);
    auto find = [&](int l, long long x, long long y) -> int {
        const int d = l - base;
        if (d < 0 || d > maxd) return -1;
        if (dense) return grid[(size_t)(off[d] + y * ((long long)nbx << d) + x)];
        auto it = at.find(key(l, x, y));
        return it == at.end() ? -1 : it->second;
    };
    double area = 0.0;
    for (int k = 0; k < n; k++) {
        const int d = lev[k] - base;
        const long long w = (long long)nbx << d, hgt = (long long)nby << d;
        if (ix[k] < 0 || iy[k] < 0 || ix[k] >= w || iy[k] >= hgt) return fail(BGF_ERR_INVALID_ARG, "block outside the domain");
        if (dense) {
            int& g = grid[(size_t)(off[d] + iy[k] * w + ix[k])];
            if (g >= 0) return fail(BGF_ERR_INVALID_ARG, "duplicate block");
            g = id[k];
        } else if (!at.emplace(key(lev[k], ix[k], iy[k]), id[k]).second) {
            return fail(BGF_ERR_INVALID_ARG, "duplicate block");
        }
        area += std::ldexp(1.0, -2 * d);
    }
    for (int k = 0; k < n; k++)  // no block may contain another
        for (long long l = lev[k] - 1, x = ix[k] >> 1, y = iy[k] >> 1; l >= base; l--, x >>= 1, y >>= 1)
            if (find((int)l, x, y) >= 0) return fail(BGF_ERR_INVALID_ARG, "overlapping blocks");
    if (area != (double)nbx * (double)nby) return fail(BGF_ERR_INVALID_ARG, "blocks do not cover the domain");
    // neighbour(s) across the side with offset (ox, oy); (f0, f1) are the
    // positions of the two finer blocks relative to 2*(x+ox, y+oy)
    auto side = [&](int k, int ox, int oy, int fx0, int fy0, int fx1, int fy1, int* first, int* second) -> bool {
        const int l = lev[k], d = l - base, me = id[k];
        const long long x = ix[k] + ox, y = iy[k] + oy;
        if (x < 0 || y < 0 || x >= ((long long)nbx << d) || y >= ((long long)nby << d)) {
            first[me] = second[me] = me;
            return true;
        }
        int nb = find(l, x, y);
        if (nb < 0 && l > base) nb = find(l - 1, x >> 1, y >> 1);
        if (nb >= 0) {
            first[me] = second[me] = nb;
            return true;
        }
        const int a = find(l + 1, 2 * x + fx0, 2 * y + fy0), c = find(l + 1, 2 * x + fx1, 2 * y + fy1);
        if (a < 0 || c < 0) return false;
        first[me] = a;
        second[me] = c;
        return true;
    };
    for (int k = 0; k < n; k++) {
        bool ok = side(k, -1, 0, 1, 0, 1, 1, LeftBot, LeftTop) && side(k, 1, 0, 0, 0, 0, 1, RightBot, RightTop) &&
                  side(k, 0, -1, 0, 1, 1, 1, BotLeft, BotRight) && side(k, 0, 1, 0, 0, 1, 0, TopLeft, TopRight);
        if (!ok) return fail(BGF_ERR_INVALID_ARG, "mesh is not 2:1 balanced");
    }
    return BGF_OK;
}

// The blocks of a multi-level mesh whose advance waits for other blocks'
// faces: those beside a finer block, and those on the domain edge when some
// boundary segment is open (edges).  nb: the eight neighbour arrays in the
// order LeftBot, LeftTop, RightBot, RightTop, TopLeft, TopRight, BotLeft,
// BotRight.  The kernels leave a finer block's shared faces to its coarser
// neighbour by what the finer block's own record says; a block list whose two
// records disagree (all) has every block wait, with all its faces stored.
template <class Nb>
inline std::vector<int> fix_blocks(const int* active, int nblk, const int* level, const Nb& nb, bool edges, bool& all,
                                   bool& odd) {
    static const int facing[8] = {2, 2, 0, 0, 6, 6, 4, 4};
    std::vector<int> list;
    all = odd = false;
    for (int k = 0; k < nblk; k++) {
        const int ib = active[k];
        bool wait = false;
        for (int q = 0; q < 8; q++) {
            const int n = nb[q][ib];
            if (level[n] > level[ib]) {
                wait = true;
                if (nb[facing[q]][n] != ib || nb[facing[q] + 1][n] != ib) all = true;
            }
            if (edges && n == ib) wait = true;
            const int n1 = nb[q & ~1][ib];
            if ((q & 1) && n1 != ib && level[n1] <= level[ib] && level[n] > level[ib]) odd = true;
        }
        if (wait) list.push_back(ib);
    }
    if (all) list.assign(active, active + nblk);
    return list;
}

// ------------------------------------------------------------ boundary segments
// A polygon (src/Input.h:107-111): closed vertex list and bounding box.
struct Polygon {
    std::vector<double> x, y;
    double xmin = 0, xmax = 0, ymin = 0, ymax = 0;
};

// A polygon from a caller's vertices as readPolygon prepares one
// (src/ReadForcing.cu:1570-1600): closed (the first vertex repeated unless the
// last equals it within 1000 epsilon), made counter-clockwise (CounterCWPoly,
// src/Poly.cu:204-237: reversed when the sum of dx*dy over its edges is
// positive), with its bounding box.
inline Polygon make_polygon(int n, const double* x, const double* y) {
    Polygon P;
    P.x.assign(x, x + n);
    P.y.assign(y, y + n);
    const double tol = std::numeric_limits<double>::epsilon() * 1000.0;
    if (!(std::fabs(P.x[0] - P.x[n - 1]) < tol && std::fabs(P.y[0] - P.y[n - 1]) < tol)) {
        P.x.push_back(P.x[0]);
        P.y.push_back(P.y[0]);
    }
    double turn = 0.0;
    for (size_t i = 0; i + 1 < P.x.size(); i++) turn = turn + (P.x[i + 1] - P.x[i]) * (P.y[i + 1] - P.y[i]);
    if (turn > 0.0) {  // reversed: the closing vertex first, then back round to it
        std::vector<double> rx(P.x.rbegin(), P.x.rend() - 1), ry(P.y.rbegin(), P.y.rend() - 1);
        rx.push_back(rx[0]);
        ry.push_back(ry[0]);
        P.x.swap(rx);
        P.y.swap(ry);
    }
    P.xmin = *std::min_element(P.x.begin(), P.x.end());
    P.xmax = *std::max_element(P.x.begin(), P.x.end());
    P.ymin = *std::min_element(P.y.begin(), P.y.end());
    P.ymax = *std::max_element(P.y.begin(), P.y.end());
    return P;
}

// The strip the side keywords pick (readbndpolysegment, src/ReadForcing.cu:796-866):
// 2*eps wide along side s (0 left, 1 right, 2 bottom, 3 top) of [xo, xmax] x [yo, ymax].
inline Polygon side_strip(int s, double xo, double xmax, double yo, double ymax, double eps) {
    const double x0 = s == 0 ? xo - eps : s == 1 ? xmax - eps : xo;
    const double x1 = s == 0 ? xo + eps : s == 1 ? xmax + eps : xmax;
    const double y0 = s == 2 ? yo - eps : s == 3 ? ymax - eps : yo;
    const double y1 = s == 2 ? yo + eps : s == 3 ? ymax + eps : ymax;
    Polygon P;
    P.x = {x0, x1, x1, x0, x0};
    P.y = {y0, y0, y1, y1, y0};
    P.xmin = x0; P.xmax = x1; P.ymin = y0; P.ymax = y1;
    return P;
}

// Winding number of (px, py) about P, the edge test (the cross product of the
// edge and the point) in T (wn_PnPoly, src/Poly.cu:171-189).
template <class T> inline int winding(T px, T py, const Polygon& P) {
    int wn = 0;
    for (size_t i = 0; i + 1 < P.x.size(); i++) {
        const T ax = T(P.x[i]), ay = T(P.y[i]), bx = T(P.x[i + 1]), by = T(P.y[i + 1]);
        const T side = (bx - ax) * (py - ay) - (px - ax) * (by - ay);
        if (P.y[i] <= py) {
            if (P.y[i + 1] > py && side > 0) ++wn;
        } else if (P.y[i + 1] <= py && side < 0) {
            --wn;
        }
    }
    return wn;
}

// Do the segments a0-a1 and b0-b1 meet (SegmentIntersect, src/Poly.cu:321-388):
// the parametric crossing of r = a1 - a0 and s = b1 - b0 when r x s is not
// within 1e-9 of 0; parallel segments meet only when collinear and
// overlapping, judged with the reference's product "dot" (A.x*B.x + A.x + B.y
// + A.y*B.x + A.y*B.y, src/Poly.cu:284-289), kept as the reference computes it.
inline bool segments_meet(double a0x, double a0y, double a1x, double a1y, double b0x, double b0y, double b1x,
                          double b1y) {
    const double rx = a1x - a0x, ry = a1y - a0y, sx = b1x - b0x, sy = b1y - b0y, qx = b0x - a0x, qy = b0y - a0y;
    const double rxs = rx * sy - ry * sx, qxr = qx * ry - qy * rx;
    auto dot = [](double ax, double ay, double bx, double by) { return ax * bx + ax + by + ay * bx + ay * by; };
    if (std::fabs(rxs) <= 1e-9) {
        if (std::fabs(qxr) > 1e-9) return false;
        const double rr = dot(rx, ry, rx, ry);
        const double t0 = dot(qx, qy, rx, ry) / rr, t1 = t0 + dot(sx, sy, rx, ry) / rr;
        return dot(sx, sy, rx, ry) < 0.0 ? (t0 >= 0.0 && t1 <= 1) : (t1 >= 0.0 && t0 <= 1);
    }
    const double t = (qx * sy - qy * sx) / rxs, u = qxr / rxs;
    return t >= 0.0 && t <= 1.0 && u >= 0.0 && u <= 1.0;
}

// Does block box [xo, xo + 16 dx] x [yo, yo + 16 dx] touch polygon P
// (blockinpoly, src/Poly.cu:443-504): the bounding boxes overlap, and a corner
// of the box lies in P or an edge of the box crosses an edge of P; T is the
// model's type.
template <class T> inline bool block_touches(T xo, T yo, T dx, const Polygon& P) {
    const T xr = xo + dx * 16, yt = yo + dx * 16;
    if (!(T(P.xmin) <= xr && T(P.xmax) >= xo && T(P.ymin) <= yt && T(P.ymax) >= yo)) return false;
    if (winding(xo, yo, P) || winding(xr, yo, P) || winding(xo, yt, P) || winding(xr, yt, P)) return true;
    const double bx[5] = {double(xo), double(xr), double(xr), double(xo), double(xo)};
    const double by[5] = {double(yo), double(yo), double(yt), double(yt), double(yo)};
    for (int i = 0; i < 4; i++)
        for (size_t j = 0; j + 1 < P.x.size(); j++)
            if (segments_meet(bx[i], by[i], bx[i + 1], by[i + 1], P.x[j], P.y[j], P.x[j + 1], P.y[j + 1])) return true;
    return false;
}

// The segment of each boundary block (Initbndblks, src/InitialConditions.cu:1168-1290):
// a block one of whose eight neighbours is itself belongs to the last segment
// whose polygon it touches, from its box at (Param.xo + XBlock.xo, Param.yo +
// XBlock.yo) in T, else to the remainder (index npoly); other slots get 255.
template <class T>
inline std::vector<unsigned char> assign_segments(const bgf_param& p, const std::vector<int>& active,
                                                  const std::vector<int>& level, const std::vector<double>& bxo,
                                                  const std::vector<double>& byo, const std::vector<int>* nb,
                                                  const std::vector<Polygon>& polys, int cap) {
    std::vector<unsigned char> seg(cap, 255);
    const int npoly = (int)polys.size();
    for (int ib : active) {
        bool bnd = false;
        for (int k = 0; k < 8; k++) bnd = bnd || nb[k][ib] == ib;
        if (!bnd) continue;
        const T dxlev = calcres_t(T(p.dx), level[ib]);
        const T xo = T(p.xo + (double)T(bxo[ib])), yo = T(p.yo + (double)T(byo[ib]));
        int s = npoly;
        for (int k = 0; k < npoly; k++)
            if (block_touches(xo, yo, dxlev, polys[k])) s = k;
        seg[ib] = (unsigned char)s;
    }
    return seg;
}

}  // namespace bgf_host
