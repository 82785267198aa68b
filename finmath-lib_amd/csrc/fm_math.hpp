// Double-precision natural logarithm for the path kernels.
//
// x = m 2^e with m in [sqrt(1/2), sqrt(2)), f = m - 1 (exact), s = f / (2 + f):
//   log(1 + f) = 2 atanh(s) = f - s (f - R),   R = sum_{k>=1} 2/(2k+1) s^(2k)
// evaluated as f - (h - s (h + R)) with h = f^2/2 (the identity f (1 - s) = 2 s turns
// f - s f into f - h + s h), and log(x) = e ln2_hi + (log(1 + f) + e ln2_lo) with ln2_hi
// holding 21 significant bits so that e ln2_hi is exact. |s| <= 0.1716, so ten terms of
// the series leave a truncation below 1e-18 relative; the error of the result is about
// one unit in the last place (checked against the C library on the CPU).
//
// Fused multiply-adds are written explicitly, so the result does not depend on the
// translation unit's contraction setting.
#pragma once

#include <hip/hip_runtime.h>
#include <cmath>

namespace fm {

__host__ __device__ inline double fm_log(double x) {
    constexpr double kLn2Hi = 0x1.62e42p-1;                  // 21 significant bits of ln 2
    constexpr double kLn2Lo = 0x1.fdf473de6af28p-22;         // ln 2 - kLn2Hi
    constexpr double kSqrtHalf = 0.70710678118654752440;
    int e = 0;
    double m = frexp(x, &e);                                 // x = m 2^e, m in [0.5, 1)
    if (m < kSqrtHalf) { m = m + m; e = e - 1; }
    const double f = m - 1.0;
    const double d = 2.0 + f;
    double s = f / d;
    const double z = s * s;
    // R(z) = z (2/3 + z (2/5 + z (2/7 + ... + z 2/21)))
    double p = 0.09523809523809523;                          // 2/21
    p = fma(p, z, 0.10526315789473684);                      // 2/19
    p = fma(p, z, 0.11764705882352941);                      // 2/17
    p = fma(p, z, 0.13333333333333333);                      // 2/15
    p = fma(p, z, 0.15384615384615385);                      // 2/13
    p = fma(p, z, 0.18181818181818182);                      // 2/11
    p = fma(p, z, 0.22222222222222222);                      // 2/9
    p = fma(p, z, 0.2857142857142857);                       // 2/7
    p = fma(p, z, 0.4);                                      // 2/5
    p = fma(p, z, 0.6666666666666666);                       // 2/3
    const double R = p * z;
    const double h = 0.5 * f * f;
    const double de = (double)e;
    const double r = de * kLn2Hi + (f - (h - fma(s, h + R, de * kLn2Lo)));
    // x <= 0, infinities and NaN: log(0) = -inf, log(x < 0) = NaN, log(+inf) = +inf
    if (!(x > 0.0) || x == HUGE_VAL) return (x == 0.0) ? -HUGE_VAL : ((x > 0.0) ? x : (x - x) / (x - x));
    return r;
}

// 1 / b by the hardware reciprocal estimate refined with two Newton-Raphson steps (r <- r + r (1 - b r)),
// and a / b from it with one correction of the quotient (q <- q + r (a - b q)). For finite b of
// moderate exponent (the path kernels divide by 1 + L d or L + 1/d) the quotient is within one unit
// in the last place of the correctly rounded one and almost always equal to it; b = +-inf gives NaN
// instead of zero. Seven instructions against the eleven of the scaled IEEE division sequence, and
// numerators with one divisor share the reciprocal.
__device__ __forceinline__ double fm_rcp_nr(double b) {
    double r = __builtin_amdgcn_rcp(b);
    double e = fma(-b, r, 1.0);
    r = fma(r, e, r);
    e = fma(-b, r, 1.0);
    return fma(r, e, r);
}

__device__ __forceinline__ double fm_div_nr_r(double a, double b, double r) {
    const double q = a * r;
    return fma(r, fma(-b, q, a), q);
}

// The coefficients of fm_exp2 in scalar registers, made once before a kernel's loops (an FP64 operand
// cannot be a literal on this target). The empty asm hides their values: as known constants the
// compiler copies each into vector registers for an accumulating multiply-add, two moves more per
// Horner step.
struct Exp2Coef {
    double c1, c2, c3, c4, c5, c6, c7, c8, c9, c10, c11;
    __device__ __forceinline__ Exp2Coef()
        : c1(0x1.62e42fefa39f3p-1), c2(0x1.ebfbdff82c598p-3), c3(0x1.c6b08d7048f31p-5), c4(0x1.3b2ab6fba1e1cp-7),
          c5(0x1.5d87fe7bbbe09p-10), c6(0x1.43091309610fcp-13), c7(0x1.ffcbee3b0a61cp-17), c8(0x1.62bfd49ededd3p-20),
          c9(0x1.b54167a1b0034p-24), c10(0x1.e605f964b639dp-28), c11(0x1.c063841f3a21dp-32) {
#if defined(__HIP_DEVICE_COMPILE__)
        asm("" : "+s"(c1), "+s"(c2), "+s"(c3), "+s"(c4), "+s"(c5), "+s"(c6));
        asm("" : "+s"(c7), "+s"(c8), "+s"(c9), "+s"(c10), "+s"(c11));
#endif
    }
};

// 2^x. x = n + r with n the nearest integer (both exact), 2^r = 1 + r q(r) with q the minimax
// polynomial of degree 10 on [-1/2, 1/2] (Remez exchange in 60-digit arithmetic; relative error of 2^r
// below 1.8e-17, below 4.3e-17 with the coefficients rounded to double), scaled by ldexp, which also gives
// the underflow to zero and the overflow to infinity: within one unit in the last place. NaN
// propagates; an infinite x gives NaN, so a state that stands for log2(0) is held as a finite
// number whose power underflows instead.
__device__ __forceinline__ double fm_exp2(double x, const Exp2Coef& k) {
    const double n = __builtin_rint(x);
    const double r = x - n;
    double p = fma(k.c11, r, k.c10);
    p = fma(p, r, k.c9);
    p = fma(p, r, k.c8);
    p = fma(p, r, k.c7);
    p = fma(p, r, k.c6);
    p = fma(p, r, k.c5);
    p = fma(p, r, k.c4);
    p = fma(p, r, k.c3);
    p = fma(p, r, k.c2);
    p = fma(p, r, k.c1);
    p = fma(p, r, 1.0);
    return __builtin_amdgcn_ldexp(p, (int)n);
}

} // namespace fm
