// Double-double arithmetic (an unevaluated sum hi + lo of two doubles, about
// 106 bits) from the error-free transformations of Dekker and Knuth.
// Contraction is off: the error terms depend on the exact operation order.
#pragma once
#include <hip/hip_runtime.h>

namespace mcmb {

struct dd {
    double hi, lo;
};

// s + e = a + b exactly (two_sum), for |a| >= |b| (quick_two_sum)
__device__ __forceinline__ dd two_sum(double a, double b)
{
#pragma clang fp contract(off)
    const double s = a + b, t = s - a;
    return dd{s, (a - (s - t)) + (b - t)};
}
__device__ __forceinline__ dd quick_two_sum(double a, double b)
{
#pragma clang fp contract(off)
    const double s = a + b;
    return dd{s, b - (s - a)};
}
__device__ __forceinline__ dd two_prod(double a, double b)
{
#pragma clang fp contract(off)
    const double p = a * b;
    return dd{p, __builtin_fma(a, b, -p)};
}
__device__ __forceinline__ dd operator+(dd a, dd b)
{
#pragma clang fp contract(off)
    const dd s = two_sum(a.hi, b.hi), t = two_sum(a.lo, b.lo);
    const dd u = quick_two_sum(s.hi, s.lo + t.hi);
    return quick_two_sum(u.hi, u.lo + t.lo);
}
__device__ __forceinline__ dd operator-(dd a) { return dd{-a.hi, -a.lo}; }
__device__ __forceinline__ dd operator-(dd a, dd b) { return a + (-b); }
__device__ __forceinline__ dd operator*(dd a, dd b)
{
#pragma clang fp contract(off)
    const dd p = two_prod(a.hi, b.hi);
    return quick_two_sum(p.hi, __builtin_fma(a.lo, b.hi, __builtin_fma(a.hi, b.lo, p.lo)));
}
__device__ __forceinline__ dd operator*(double a, dd b)
{
#pragma clang fp contract(off)
    const dd p = two_prod(a, b.hi);
    return quick_two_sum(p.hi, __builtin_fma(a, b.lo, p.lo));
}
__device__ __forceinline__ dd operator/(dd a, dd b)
{
#pragma clang fp contract(off)
    const double q = a.hi / b.hi;
    const dd r = a - q * b;
    const double q2 = r.hi / b.hi;
    const dd r2 = r - q2 * b;
    return quick_two_sum(q, q2) + dd{r2.hi / b.hi, 0.0};
}
// Sums with a biased high part: acc.hi starts at B = 3 2^k with 2^k above the
// sum of the terms' magnitudes, so it stays in one binade (of unit u =
// 2^(k-51)) throughout.  acc.hi + a b.hi rounded to u differs from acc.hi by an
// exact multiple of u, which the next operation recovers, and the term's rest,
// at most u / 2, goes to acc.lo with b's low part: five operations a term (six
// for two dd), against eleven with an error-free sum of the running value.  A
// term rounds at 2^-53 of acc.lo: of rests of random sign that is about 2^-104
// of 2^k a term, but acc.lo is not folded back, and after n rests of one sign it
// is n u / 2 and the sum's error up to n^2 2^-104 of 2^k.
__device__ __forceinline__ double dd_bias(double bound)
{
    return bound > 0.0 && bound < INFINITY ? ldexp(3.0, ilogb(bound) + 1) : 3.0;
}
// acc += a b, a double
__device__ __forceinline__ void dd_bmac(dd& acc, double a, dd b)
{
#pragma clang fp contract(off)
    const double s = __builtin_fma(a, b.hi, acc.hi), p = s - acc.hi;
    acc.hi = s;
    acc.lo = __builtin_fma(a, b.lo, acc.lo) + __builtin_fma(a, b.hi, -p);
}
__device__ __forceinline__ void dd_bmac(dd& acc, dd a, dd b)
{
#pragma clang fp contract(off)
    const double s = __builtin_fma(a.hi, b.hi, acc.hi), p = s - acc.hi;
    acc.hi = s;
    acc.lo = __builtin_fma(a.lo, b.hi, __builtin_fma(a.hi, b.lo, acc.lo)) + __builtin_fma(a.hi, b.hi, -p);
}
// the sum of a biased accumulator
__device__ __forceinline__ dd dd_unbias(dd a, double B) { return two_sum(a.hi - B, a.lo); }
// (by components: a ?: of two dd selects an address, which keeps both in memory)
__device__ __forceinline__ dd dd_sel(bool c, dd a, dd b) { return dd{c ? a.hi : b.hi, c ? a.lo : b.lo}; }
__device__ __forceinline__ dd dd_shfl_xor(dd a, int o) { return dd{__shfl_xor(a.hi, o), __shfl_xor(a.lo, o)}; }

}  // namespace mcmb
