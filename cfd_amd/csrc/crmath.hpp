// Division, square root and the two powers the path needs, in binary64.
//
// Division and square root are the correctly rounded ones ('/' and sqrt()
// give the same bits) without the compiler's scaling steps for operands near
// the ends of the exponent range, and with the parts that several quotients
// share formed once:
//   recip(b)       Newton's iteration on the hardware's reciprocal;
//   quot(a, r)     q = a r, corrected by its exact remainder a - b q (Markstein,
//                  "Computation of elementary functions on the IBM RISC
//                  System/6000 processor", 1990);
//   third(a)       a / 3 from the rounded constant 1/3, the same way;
//   sqrt_rn(x)     Goldschmidt's iteration on the hardware's reciprocal square
//                  root, corrected twice by the exact remainder x - s^2.
// Where quot is not '/': a dividend below 2^-968 (2.5e-292; its remainder is a
// multiple of 2^-106 |a| and would have to be one of 2^-1074) may give an ulp more or
// less, and a divisor of at most 2^-1024 gives an infinity for every dividend but
// zero.  Quotients that overflow, zeros, infinities and NaNs are as '/' gives them.
// Callers divide by states (density, temperature), lengths, time steps and norms
// kept above 1e-20, or a constant by a sum of velocities (where '/' overflows too);
// a dividend that small is a momentum or a product of velocities, far from what
// moves in a gas at rest, and its ulp is that of a velocity of 1e-292 or is lost in
// what it is added to.  On gfx950 over 1.4 10^6 pairs from all of the exponent range,
// subnormal numbers included: no other difference (third: none).
// sqrt_rn hands x below 2^-700 to sqrt().  Compared with '/' and sqrt() on gfx950
// over 5 10^8 random operands in each of five exponent ranges up to 2^+-450: no
// difference.  Instructions: '/' 11, quot 4 and recip 5, third 4; sqrt() 17,
// sqrt_rn 12.
//
// The powers are correctly rounded (round to nearest) up to a 2^-103 relative
// window around rounding midpoints, and exactly where x^(3/2) is a midpoint (x a
// square): each starts from an approximation and adds one correction carried in
// double-double with error-free products (fma):
//   x^(-1/2) = y (1 + r/2 + 3 r^2/8),   r = 1 - x y^2 (exact to 2^-103)
//   x^(3/2)  = x * sqrt(x),   sqrt(x) = s + (x - s*s) h
// with y from the hardware's reciprocal square root and one third-order step
// (relative error about 2^-52), s = sqrt(x) rounded from a value 2^-88 off, so exact
// for squares (an s an ulp off misrounds 2,772 of the 27,040 squares whose 3/2 power
// is a midpoint), and h = 1/(2 s) within an ulp.  They replace pow(x, 1.5) (calcRHS.f90:50-51, subrutinas.f90:196,400)
// and pow(x, -0.5) (subrutinas.f90:429,438-439): fewer instructions than a
// general pow, and closer to the exact value than either the device pow or
// glibc's.
#pragma once

#include <hip/hip_runtime.h>

namespace cfd {

struct Recip {
    double b, r;  // r = 1/b, within an ulp
};
__device__ __forceinline__ Recip recip(double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    r = __builtin_fma(r, __builtin_fma(-b, r, 1.0), r);
    return {b, r};
}
__device__ __forceinline__ double quot(double a, const Recip& k) {
    double q = a * k.r;
    q = __builtin_fma(__builtin_fma(-k.b, q, a), k.r, q);
    return __builtin_amdgcn_div_fixup(q, k.b, a);
}
__device__ __forceinline__ double quot(double a, double b) { return quot(a, recip(b)); }
__device__ __forceinline__ double third(double a) { return quot(a, Recip{3.0, 1.0 / 3.0}); }

// sqrt(x) for x > 2^-700, rounded from a value 2^-88 off; h: 1/(2 sqrt(x)) within 2^-44
__device__ __forceinline__ double sqrt_core(double x, double& h) {
    const double y = __builtin_amdgcn_rsq(x);
    double s = x * y;
    h = 0.5 * y;
    const double e = __builtin_fma(-h, s, 0.5);
    s = __builtin_fma(s, e, s);
    h = __builtin_fma(h, e, h);
    return __builtin_fma(__builtin_fma(-s, s, x), h, s);
}
__device__ __forceinline__ double sqrt_rn(double x) {
    if (__any(x < 0x1p-700 && x != 0.0)) return sqrt(x);
    double h;
    double s = sqrt_core(x, h);
    s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
    return x == 0.0 || x == __builtin_huge_val() ? x : s;
}

// x^(-1/2) to about an ulp (0, infinities, NaN as 1/sqrt(x) gives them in *edge)
__device__ __forceinline__ double rsqrt_near(double x, double* edge) {
    const double y = __builtin_amdgcn_rsq(x);
    *edge = y;
    const double e = __builtin_fma(-(x * y), y, 1.0);
    return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

__device__ __forceinline__ double pow_3_2(double x) {
    double h;
    const double s = sqrt_core(x, h);
    h = __builtin_fma(h, __builtin_fma(-h, s, 0.5), h);
    const double sl = __builtin_fma(-s, s, x) * h;  // sqrt(x) = s + sl
    const double p = x * s;
    const double pe = __builtin_fma(x, s, -p);  // x*s = p + pe, exact
    const double r = p + (pe + x * sl);
    return (x == 0.0 || !(x < __builtin_huge_val())) ? x * x : r;
}

__device__ __forceinline__ double pow_m1_2(double x) {
    double edge;
    const double y = rsqrt_near(x, &edge);
    const double p = y * y, pe = __builtin_fma(y, y, -p);   // y^2 = p + pe
    const double q = x * p, qe = __builtin_fma(x, p, -q);   // x p = q + qe
    const double r = ((1.0 - q) - qe) - x * pe;             // 1 - x y^2
    const double z = y + y * (r * __builtin_fma(r, 0.375, 0.5));
    // 0 -> inf, inf -> 0, NaN -> NaN as pow(x, -0.5) gives for x >= 0
    return (x == 0.0 || !(x < __builtin_huge_val())) ? edge : z;
}

}  // namespace cfd
