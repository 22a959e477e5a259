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
// result is subnormal; such a quotient is reported (div_subnormal) and divided by the caller
// again. Infinities, NaN, zeros and overflow come out as in the division.
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

// FP64 heat steps of a field whose values are all 0 or in [2^-500, 2^600): a difference of two is
// 0 or at least 2^-552, its quotient by h <= 2^50 at least 2^-602, a difference of two quotients 0
// or at least 2^-654 -- far above the 2^-969 below which the residual would not be exact -- and
// with |coef| >= 2^-100 the new value is 0 or at least 2^-908, so its magnitude shows in the high
// word, where the next step's test looks for it. div_key orders the high words so that 0 is the
// largest: a minimum over cells below kDivLow means a nonzero value under 2^-500.
constexpr unsigned kDivLow = ((1023u - 500u) << 21) - 1u;
constexpr unsigned kDivHigh = (1023u + 400u) << 21;  // at the launch's start; the steps then add at most 2^200

#if defined(__HIPCC__)
__device__ __forceinline__ unsigned div_key(double v) {  // 2 hi - 1 (the compiler takes three instructions)
    unsigned k;
    asm("v_lshl_add_u32 %0, %1, 1, -1" : "=v"(k) : "v"(__double2hiint(v)));
    return k;
}
// outside the range at the launch's start: subnormal, below 2^-500, 2^400 or more, infinite, NaN
__device__ __forceinline__ bool div_unsafe(double v) {
    const unsigned m = (unsigned)__double2hiint(v) << 1;
    return (m - kDivLow >= kDivHigh - kDivLow) && v != 0.0;
}
__device__ __forceinline__ bool div_subnormal(float q) { return __builtin_isfpclass(q, 0x90); }  // +-subnormal
#endif

// the host's side of the range: spacing, coefficient and growth of `steps` steps in `dim` dims
inline bool div_range(const double* h, int dim, double coef, int steps) {
    double g = 0;
    for (int d = 0; d < dim; ++d) {
        if (!(h[d] >= 0x1p-100 && h[d] <= 0x1p50)) return false;
        g += 4.0 * std::fabs(coef) / (h[d] * h[d]);
    }
    return std::fabs(coef) >= 0x1p-100 && std::fabs(coef) <= 0x1p200 && steps * std::log2(1.0 + g) <= 200.0;
}

}  // namespace opf
