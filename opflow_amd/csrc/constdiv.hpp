// Correctly rounded division by a divisor known before the launch (a grid spacing), with the
// bits of the IEEE quotient.
//
// FP64: with y = RN(1 / h), q = RN(x y) and the residual r = h q - x (exact in one FMA),
// RN(q - r y) is the correctly rounded x / h whenever nothing under- or overflows (Markstein,
// "Computation of elementary functions on the IBM RISC System/6000 processor", 1990; Brisebarre,
// Muller and Raina, "Accelerating correctly rounded floating-point division when the divisor is
// known in advance", IEEE Trans. Computers 53, 2004): 3 operations where the compiler's division
// takes about 11 with a quarter-rate reciprocal among them. Written with r = h q - x it keeps the
// sign of a zero x (for h > 0: a quotient by -h is minus the one by h). The callers keep x inside the safe range (div_range below).
//
// FP32: the quotient of two 24-bit numbers is at least 2^-49 (relative) away from every midpoint
// of neighbouring floats it is not equal to, and x RN64(1 / h) in FP64 is within 2^-52 of it, so
// rounding that product to float gives the IEEE quotient. It can equal a midpoint only where the
// result is subnormal, which the callers' range keeps out. Infinities, NaN, zeros and overflow come
// out as in the division.
#pragma once

#include <cmath>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define OPF_CD_HD __host__ __device__ __forceinline__
#else
#define OPF_CD_HD inline
#endif

namespace opf {

struct ConstDivisor {
    double h = 1.0, y = 1.0;  // the divisor (positive) in the field's precision, and RN64(1 / h)
};

OPF_CD_HD double const_div(double x, const ConstDivisor& c) {
    const double q = x * c.y;
    const double r = __builtin_fma(c.h, q, -x);
    return __builtin_fma(-r, c.y, q);
}
OPF_CD_HD float const_div(float x, const ConstDivisor& c) { return (float)((double)x * c.y); }

// The range of a field's values for its heat steps: every value 0 or at least 2^-T in magnitude,
// and in FP64 under 2^600.
//   FP64, T = 500: a difference of two values is 0 or at least 2^-552, its quotient by h <= 2^50 at
//   least 2^-602, a difference of two quotients 0 or at least 2^-654 -- far above the 2^-969 below
//   which the residual would not be exact -- and with |coef| >= 2^-100 the new value is 0 or at least
//   2^-908, so its magnitude shows in the high word, where the next step's test looks for it.
//   FP32, T = min(100, 101 + l, 78 + 2 l) for spacings up to 2^-l: a difference is 0 or at least
//   2^-(T + 25) (a ghost between a wall value and a cell has one or two bits below its cell), so its
//   quotient at least 2^-126; a difference of two quotients is 0 or at least 2^-(T + 48) / h, and its
//   quotient at least 2^-126 again: nothing is subnormal.
// A ghost made from a zero is its side's constant, so the constants are 0 or in the range too.
// div_key orders the magnitudes (the high words, in FP64) so that 0 is the largest: a minimum over
// cells below the key of 2^-T means that a nonzero value is smaller.
constexpr unsigned kDivLow = ((1023u - 500u) << 21) - 1u;
constexpr unsigned kDivHigh = (1023u + 400u) << 21;  // at the launch's start; the steps then add at most 2^200

#if defined(__HIPCC__)
// 2 bits - 1 in one instruction (the compiler takes three)
__device__ __forceinline__ unsigned div_key_bits(int bits) {
    unsigned k;
    asm("v_lshl_add_u32 %0, %1, 1, -1" : "=v"(k) : "v"(bits));
    return k;
}
__device__ __forceinline__ unsigned div_key(double v) { return div_key_bits(__double2hiint(v)); }
__device__ __forceinline__ unsigned div_key(float v) { return div_key_bits(__float_as_int(v)); }
// outside the range at the launch's start: subnormal, below 2^-500, 2^400 or more, infinite, NaN
__device__ __forceinline__ bool div_unsafe(double v) {
    const unsigned m = (unsigned)__double2hiint(v) << 1;
    return (m - kDivLow >= kDivHigh - kDivLow) && v != 0.0;
}
#endif

// T of FP32 for spacings h[0 .. dim - 1]
inline int div_exp32(const double* h, int dim) {
    int l = 1000, e;
    for (int d = 0; d < dim; ++d) {
        std::frexp(h[d], &e);  // h < 2^e
        if (-e < l) l = -e;
    }
    int t = 100;
    if (101 + l < t) t = 101 + l;
    if (78 + 2 * l < t) t = 78 + 2 * l;
    return t;
}
// the least key of a value in the range of spacings h[0 .. dim - 1]
inline unsigned div_low(const double* h, int dim, bool f64) {
    if (f64) return kDivLow;
    const int t = div_exp32(h, dim);
    return t < -100 ? 0xffffffffu : ((unsigned)(127 - t) << 24) - 1u;
}
// a side's constant: the wall's value, or what a slope adds to the cell's
inline bool div_side(double c, const double* h, int dim, bool f64) {
    c = std::fabs(c);
    return c == 0.0 || (f64 ? c >= 0x1p-400 && c <= 0x1p400 : c >= std::ldexp(1.0, -div_exp32(h, dim)));
}

// the host's side of the range: spacing, coefficient and growth of `steps` steps in `dim` dims
inline bool div_range(const double* h, int dim, double coef, int steps, bool f64) {
    double g = 0;
    for (int d = 0; d < dim; ++d) {
        if (!(f64 ? h[d] >= 0x1p-100 && h[d] <= 0x1p50 : h[d] >= 0x1p-60 && h[d] <= 0x1p20)) return false;
        g += 4.0 * std::fabs(coef) / (h[d] * h[d]);
    }
    return !f64 || (std::fabs(coef) >= 0x1p-100 && std::fabs(coef) <= 0x1p200 && steps * std::log2(1.0 + g) <= 200.0);
}

}  // namespace opf
