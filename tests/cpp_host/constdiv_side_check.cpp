// FP32 ghosts of a zero cell beside a wall value or slope (constdiv.hpp): the quotient through the
// reciprocal has the bits of the division for every constant that div_side takes, and for those
// midway between two subnormal floats, where it would not, div_side refuses them.
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>

#include "constdiv.hpp"

int main() {
    std::mt19937_64 g(5);
    long long n = 0, taken = 0, off = 0;
    for (double h : {196., 300., 308., 392., 12., 7., 1.3, 0.3, 1. / 300, 1000., 65537., 1048575., 1e-9})
        for (int q = 0; q < 200000; ++q) {
            // wall values whose ghost quotient is near an integer and a half of the least float, up to
            // ordinary ones
            const double v = q % 2 ? std::ldexp((double)(2 * (g() % (1u << 22)) + 1), -151)
                                   : std::ldexp(1.0 + (double)(g() % (1u << 23)) * 0x1p-23, (int)(g() % 150) - 140);
            const float c2 = (float)(h * v), c3 = (float)(h / 2);  // the rule (c1 u - c2) / c3 at u = 0
            const opf::ConstDivisor d{(double)c3, 1.0 / (double)c3};
            const float x = 0.0f - c2, want = x / c3, got = opf::const_div(x, d);
            const bool same = std::memcmp(&want, &got, 4) == 0, ok = opf::div_side((double)c2 / (double)c3, &h, 1, false);
            ++n;
            taken += ok;
            off += !same;
            if (ok && !same) return std::printf("h %a wall %a: %a, not %a\n", h, v, got, want), 1;
            // the difference to a zero cell over h, as the next step forms it
            const opf::ConstDivisor s{(double)(float)h, 1.0 / (double)(float)h};
            const float dw = want / (float)h, dg = opf::const_div(want, s);
            if (ok && std::memcmp(&dw, &dg, 4)) return std::printf("h %a ghost %a: %a, not %a\n", h, want, dg, dw), 1;
        }
    if (!opf::div_side(0.0, &(const double&)1.3, 1, false) || taken < n / 20 || off < 100)
        return std::printf("taken %lld of %lld, %lld differ\n", taken, n, off), 1;
    std::printf("passed %lld\n", n);
    return 0;
}
