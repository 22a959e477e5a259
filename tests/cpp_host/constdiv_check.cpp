// const_div (constdiv.hpp) against the IEEE division: random and hard significands over the
// exponents its callers keep to, signed zeros, and for float every kind of value.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>

#include "constdiv.hpp"

using opf::ConstDivisor;
static std::mt19937_64 g(7);

static double make(uint64_t mant, int e, bool neg) {
    return std::ldexp(1.0 + (double)(mant & ((1ull << 52) - 1)) * 0x1p-52, e) * (neg ? -1 : 1);
}
template <typename T>
static bool same(T a, T b) {
    return std::memcmp(&a, &b, sizeof(T)) == 0 || (a != a && b != b);
}

// x / h as the callers form it: a quotient by a negative divisor is minus the one by its absolute value
template <typename T>
static T quotient(T x, T h) {
    const ConstDivisor c{std::fabs((double)h), 1.0 / std::fabs((double)h)};
    return h < 0 ? -opf::const_div(x, c) : opf::const_div(x, c);
}

int main() {
    long long n = 0;
    // FP64: spacings 1 / n, and random ones with significands near the ends of the binade
    for (int d = 0; d < 600; ++d) {
        double h = d < 300 ? 1.0 / (3 + 7 * d) : make(d % 3 == 0 ? g() : d % 3 == 1 ? g() % 64 : ~(g() % 64), -(int)(g() % 40), false);
        if (d % 5 == 0) h = -h;
        for (int q = 0; q < 8000; ++q) {
            const uint64_t m = q % 3 == 0 ? g() : q % 3 == 1 ? g() % 256 : ~(g() % 256);
            const double x = make(m, (int)(g() % 1500) - 850, g() & 1);
            if (!same(quotient(x, h), x / h)) return std::printf("f64 %a / %a\n", x, h), 1;
            // quotients next to a rounding boundary: x within an ulp of (q + half ulp) h
            const double b = std::nextafter(x / h * h, q & 1 ? 1e300 : -1e300);
            if (!same(quotient(b, h), b / h)) return std::printf("f64 %a / %a\n", b, h), 1;
            n += 2;
        }
        for (double z : {0.0, -0.0})
            if (!same(quotient(z, h), z / h)) return std::printf("zero / %a\n", h), 1;
    }
    // float: every significand at one exponent, and random bit patterns (subnormal quotients are
    // the caller's)
    for (float h : {1.f / 300, 1.f / 260, 1.f / 7, 0.3f, 1.f / 3, 1.9999999f, 1.0000001f, -0.0123f}) {
        auto check = [&](float x) {
            const float q = x / h;
            if (std::fpclassify(q) == FP_SUBNORMAL || (q == 0 && x != 0)) {
                // the product rounds to a neighbour at most, so the caller sees a subnormal or 0
                const int k = std::fpclassify(quotient(x, h));
                return k == FP_SUBNORMAL || same(quotient(x, h), q) || std::fabs(quotient(x, h)) == 0x1p-126f;
            }
            ++n;
            return same(quotient(x, h), q);
        };
        for (uint32_t m = 0; m < (1u << 23); m += 3) {
            const uint32_t b = 0x3f800000u | m;
            float x;
            std::memcpy(&x, &b, 4);
            if (!check(x)) return std::printf("f32 %a / %a\n", x, h), 1;
        }
        for (int q = 0; q < 2000000; ++q) {
            const uint32_t b = (uint32_t)g();
            float x;
            std::memcpy(&x, &b, 4);
            if (!check(x)) return std::printf("f32 %a / %a\n", x, h), 1;
        }
    }
    // the range test of the host
    const double h3[3] = {1. / 300, 1. / 260, 1. / 220}, bad[3] = {1e-40, 1., 1.};
    if (!opf::div_range(h3, 3, 1e-6, 128, true) || opf::div_range(bad, 3, 1e-6, 3, true) ||
        opf::div_range(h3, 3, 1e-50, 3, true) || opf::div_range(h3, 3, 1e30, 128, true))
        return std::printf("div_range\n"), 1;
    std::printf("passed %lld\n", n);
    return 0;
}
