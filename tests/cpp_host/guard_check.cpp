// The guarded division of compiled sweeps (guard_device.inc) on the host: every numerator from 0 to
// beyond the guard's lower bound either has the bits of the IEEE quotient or is reported to the redo,
// and neither a zero nor an ordinary numerator is.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <random>

#define __device__
#define __forceinline__ inline
using std::max;
using std::min;
static int __double2hiint(double v) {
    int64_t b;
    std::memcpy(&b, &v, 8);
    return (int)(b >> 32);
}
static unsigned opf_key_bits(int v) { return ((unsigned)v << 1) - 1u; }
#define OPF_SHARED_SRC(...) __VA_ARGS__
#include "guard_device.inc"

int main() {
    std::mt19937_64 g(11);
    long long n = 0;
    for (double h : {1.35, 1.7, 1.3, 3.3, 7.7, 3., 7., 49., 98., 1.9999999999999998, 1.0000000000000002, 0.1, 1. / 300, 1e-30, 1e30}) {
        auto check = [&](double x) {
            unsigned lo = 0xffffffffu, lob = lo;
            int hi = 0;
            const double q = opf_cdiv(lo, x, h, 1.0 / h), r = opf_cdivb(lob, hi, x, h, 1.0 / h), want = x / h;
            ++n;
            if (lo != lob || std::memcmp(&q, &r, 8)) return std::printf("forms %a / %a\n", x, h), false;
            if (opf_low(lo) ? x == 0 || std::fabs(x) >= 0x1p-600 : std::memcmp(&q, &want, 8) != 0)
                return std::printf("%a / %a: %a, not %a\n", x, h, q, want), false;
            return true;
        };
        for (int k = 0; k < 20000; ++k)
            for (int s : {1, -1})
                if (!check(s * k * 0x1p-1074)) return 1;
        for (int e = -1075; e < 700; ++e)  // around every power of two, and anywhere between
            for (int q = 0; q < 60; ++q) {
                const uint64_t m = q % 3 == 0 ? g() >> 12 : q % 3 == 1 ? g() % 64 : (1ull << 52) - 1 - g() % 64;
                if (!check(std::ldexp(1.0 + (double)m * 0x1p-52, e) * (q & 1 ? -1 : 1))) return 1;
            }
        if (!check(0.0) || !check(-0.0)) return 1;
    }
    std::printf("passed %lld\n", n);
    return 0;
}
