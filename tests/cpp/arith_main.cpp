// Host check of bgf_arith.h against the divisions that it stands for.  Prints
// the number of results that differ and the first of them; exits 1 if any do.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <vector>

#include "bgf_arith.h"

static long wrong = 0;

template <class T> void expect(const char* what, T got, T want, T a, T b) {
    if (got == want || (got != got && want != want)) return;
    if (!wrong++) std::printf("%s: %a, not %a, of %a and %a\n", what, (double)got, (double)want, (double)a, (double)b);
}

// Every FP32 significand, from the rounded reciprocal and its neighbours; with
// a significand of ones from the rounded reciprocal, which the hardware gives.
static void reciprocals_fp32() {
    for (uint32_t e : {103u, 126u, 127u, 150u})
        for (uint32_t m = 0; m < 1u << 23; m++) {
            const uint32_t bits = e << 23 | m;
            float b;
            std::memcpy(&b, &bits, 4);
            const float r = 1.0f / b;
            expect("rcp", bgf::rounded_rcp(b, r), r, b, r);
            if (m == (1u << 23) - 1) continue;
            for (float y : {std::nextafter(r, 0.0f), std::nextafter(r, INFINITY)})
                expect("rcp", bgf::rounded_rcp(b, y), r, b, y);
        }
}

static void reciprocals_fp64() {
    std::mt19937_64 rng(5);
    for (long k = 0; k < 2000000; k++) {
        // significands at random, and near both ends of the binade
        uint64_t m = rng() >> 12;
        if (k % 4 == 1) m &= 0xff;
        if (k % 4 == 2) m |= ((uint64_t(1) << 52) - 1) ^ 0xff;
        if (m == (uint64_t(1) << 52) - 1) continue;
        const uint64_t bits = (uint64_t)(1023 - 40 + k % 80) << 52 | m;
        double b;
        std::memcpy(&b, &bits, 8);
        const double r = 1.0 / b, off = std::ldexp((double)(int64_t)rng(), -63 - 22);
        expect("rcp", bgf::rounded_rcp(b, r * (1.0 + off)), r, b, off);
    }
    for (int e = -60; e < 60; e++) {
        const double b = std::ldexp(2.0 - 0x1p-52, e);
        expect("rcp", bgf::rounded_rcp(b, 1.0 / b), 1.0 / b, b, b);
    }
}

template <class T> T any(std::mt19937_64& rng) {
    T x;
    const uint64_t v = rng();
    std::memcpy(&x, &v, sizeof(T));
    return x;
}

template <class T> void fixed_divisions() {
    std::mt19937_64 rng(6);
    const T one = 1, ones = std::nextafter(T(2), one), inf = std::numeric_limits<T>::infinity();
    std::vector<T> ds = {one / 3, 10, T(9.99), 40, 20, ones, std::nextafter(one, T(2)), T(0x1p-20), T(0x1p20), T(0x1p-21), T(3e6), T(1e-4),
                         T(0x1p-60)};
    for (T d : ds) {
        const bgf::FixedDiv<T> K = bgf::fixed_div(d);
        auto check = [&](T x) {
            expect("fixed division", bgf::odd_div(K, x) ? x / d : bgf::quick_div(K, x), x / d, x, d);
        };
        for (int k = 0; k < 400000; k++) {
            check(any<T>(rng));                                                   // any bits
            check(std::ldexp(T((double)(int64_t)rng() * 0x1p-63), (int)(rng() % 60) - 50));  // ordinary differences
        }
        const T den = std::numeric_limits<T>::denorm_min(), mx = std::numeric_limits<T>::max();
        for (T x : {T(0), -T(0), K.lo, K.hi, std::nextafter(K.lo, T(0)), std::nextafter(K.hi, inf), den, mx, -mx, inf, -inf,
                    inf - inf})
            check(x);
    }
}

int main() {
    reciprocals_fp32();
    reciprocals_fp64();
    fixed_divisions<float>();
    fixed_divisions<double>();
    std::printf("%ld wrong\n", wrong);
    return wrong != 0;
}
