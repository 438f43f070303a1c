// Correctly rounded FP64 quotients and square roots that share their reciprocals, from the
// fused-multiply-add iterations of P. Markstein ("Computation of elementary functions on the IBM RISC
// System/6000 processor", IBM J. Res. Dev. 34 (1990) 111): with y the correctly rounded reciprocal of b
// and q within an ulp or two of a / b, q + (a - b q) y rounded once is the correctly rounded quotient.
// A pair of the FP64 sums divides three times by its distance and twice by its mean density; one
// reciprocal serves each, where a division of its own per quotient repeats the reciprocal and adds the
// scaling of extreme operands.  Valid for operands whose reciprocal, square, quotient and remainder are
// normal numbers; the callers keep others on the plain operators (quot_holds; a coordinate difference below
// 1e-290 in a unit vector may round the other way).
//
// y0 is a seed of at least 20 good bits: the hardware's approximation, or any other in a host test.
#pragma once

#include <cmath>

namespace sphfem {

#if defined(__HIPCC__)
#define SPHFEM_HD __host__ __device__ __forceinline__
#else
#define SPHFEM_HD inline
#endif

// a divisor and its reciprocal, by recip_from within an ulp of the correctly rounded one.  With that
// reciprocal the quotients are correctly rounded, but for dividends that are powers of two by a divisor
// whose fraction bits are all ones (where 1 / b lies 2^-106 beyond the middle of two numbers).
struct Recip {
    double b, y;
};

// two Newton steps: 20 -> 40 -> 80 good bits, the second rounded once
SPHFEM_HD Recip recip_from(double b, double y0) {
    const double y = std::fma(std::fma(-b, y0, 1.), y0, y0);
    return {b, std::fma(std::fma(-b, y, 1.), y, y)};
}

// the correctly rounded reciprocal, from a seed of at least 40 good bits: the first step ends within an ulp,
// and the second then rounds correctly for every divisor but one with all ones (Markstein), which is divided
// out.  The upper fraction bits select a few divisors more.
SPHFEM_HD Recip recip_rounded(double b, double y0) {
    Recip r = recip_from(b, y0);
    unsigned long long bits;
    __builtin_memcpy(&bits, &b, 8);
    if (((bits >> 32) & 0xfffff) == 0xfffff) r.y = 1. / b;
    return r;
}

SPHFEM_HD double quot(double a, const Recip &r) {
    const double q = a * r.y;
    return std::fma(std::fma(-r.b, q, a), r.y, q);
}

// whether quot() holds for dividend a by a divisor of 1e-100 to 1e100: a has an exponent of 2^-600 to 2^600,
// so that quotient and remainder are normal numbers (it is not zero, subnormal, near overflow or non-finite)
SPHFEM_HD bool quot_holds(double a) {
    unsigned long long bits;
    __builtin_memcpy(&bits, &a, 8);
    return ((unsigned)(bits >> 52) & 0x7ff) - (1023u - 600u) <= 1200u;
}

// square root of x and the half reciprocal root the iteration carries (h = 1 / (2 sqrt(x)) to 40 bits)
SPHFEM_HD double sqrt_from(double x, double y0, double &h) {
    double g = x * y0;
    h = 0.5 * y0;
    const double r = std::fma(-h, g, 0.5);
    g = std::fma(g, r, g);
    h = std::fma(h, r, h);
    g = std::fma(std::fma(-g, g, x), h, g);
    return std::fma(std::fma(-g, g, x), h, g);
}

// single-precision root of a radicand that is a single-precision number: the double root rounded to
// single precision is the correctly rounded single root (53 >= 2 * 24 + 2 bits), so it needs no final
// correction; h as above
SPHFEM_HD double sqrtf_from(double x, double y0, double &h) {
    double g = x * y0;
    h = 0.5 * y0;
    const double r = std::fma(-h, g, 0.5);
    g = std::fma(g, r, g);
    h = std::fma(h, r, h);
    return (double)(float)std::fma(std::fma(-g, g, x), h, g);
}

}  // namespace sphfem
