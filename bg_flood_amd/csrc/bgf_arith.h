// bgf_arith.h -- divisions by multiply-adds with the rounding of IEEE
// division, for the kernels and for host tests of them.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>

namespace bgf {

using std::fma;

// Division by a fixed d with the rounding of an IEEE division, in four
// multiply-adds instead of its eleven instructions (of which the reciprocal
// alone takes the time of four): with zh = RN(1/d) and zl the rest of 1/d,
// q0 = RN(x zh + RN(x zl)) is within an ulp of x/d, the remainder r = x - d q0
// is exact in a multiply-add, and RN(q0 + r zh) is the correctly rounded
// quotient (Markstein, IBM J. Res. Dev. 34, 1990; the two-part reciprocal is
// that of Brisebarre and Muller).  That needs x to be zero or between lo and
// hi, well inside the normal range, and d in [2^-20, 2^20]; other x (the
// numerical precursors of a wave reach such sizes) are `odd` and take the
// division itself.
template <class T> struct FixedDiv {
    T d, zh, zl, lo, hi;
};
__host__ __device__ inline void fixed_div_range(float& lo, float& hi) { lo = 0x1p-100f; hi = 0x1p100f; }
__host__ __device__ inline void fixed_div_range(double& lo, double& hi) { lo = 0x1p-960; hi = 0x1p960; }
template <class T> __host__ __device__ inline FixedDiv<T> fixed_div(T d) {
    FixedDiv<T> K;
    K.d = d;
    K.zh = T(1.0) / d;
    K.zl = fma(-d, K.zh, T(1.0)) * K.zh;
    fixed_div_range(K.lo, K.hi);
    if (!(d >= T(0x1p-20) && d <= T(0x1p20))) K.hi = T(-1.0);  // every x is odd
    return K;
}
template <class T> __host__ __device__ inline bool odd_div(const FixedDiv<T>& K, T x) {
    const T a = fabs(x);
    return (a < K.lo && x != T(0.0)) || a > K.hi;
}
template <class T> __host__ __device__ inline T quick_div(const FixedDiv<T>& K, T x) {
    const T q = fma(x, K.zh, x * K.zl);
    return fma(fma(-K.d, q, x), K.zh, q);
}
// 1 / b rounded as IEEE division rounds it, for b of ordinary size (here the
// spread of a face's wave speeds, above epsilon wherever the result is used),
// from y near 1 / b (in FP32 to an ulp): Newton steps and Markstein's
// correction, without the scaling that extreme operands need.
//
// The correction has one exception, a significand of b of ones: 1 / b lies
// just above the middle between a power of two and its successor, and from the
// power of two the last sum is a tie, which returns it.  There the result is
// right if y is the successor already, and on gfx950 it is: v_rcp_f32 rounds
// this divisor as division does, and v_rcp_f64 returns the division's result
// (both measured, FP32 over all significands at eleven exponents with 10.7 % of
// the y off by an ulp, FP64 at 128 exponents; every result was the division's).
template <class T> __host__ __device__ inline T rounded_rcp(T b, T y) {
    y = fma(fma(-b, y, T(1.0)), y, y);
    y = fma(fma(-b, y, T(1.0)), y, y);
    return fma(fma(-b, y, T(1.0)), y, y);
}

}  // namespace bgf
