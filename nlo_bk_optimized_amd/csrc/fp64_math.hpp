// FP64 logarithm, exponential, reciprocal and quotient for arguments that are
// known to be ordinary numbers.  The library's forms cover every input (zeros,
// subnormal and infinite values, NaN) and carry the logarithm in
// double-double: 98 instructions for log, 175 for log1p(exp(-x)), 12 for a
// quotient, which made most of what the BK integrands in FP64 issue.  Here: 39,
// 24 (log1p_fold64 from a power) and 6.  The fixed K1 rule on 1024 nodes went
// from 2.63 to 1.91 ms, on the default grid of 101 from 85 to 54 us with them,
// one RHS of the adaptive rule on 256 nodes from 1.96 to 1.59 ms.  Errors over
// 2^22 arguments, largest / mean, in ulp: log64 0.65 / 0.250 (the library's log
// 0.64 / 0.252), exp64 0.75 / 0.254 (0.87 / 0.256), rcp64 and div64 0.50.
#pragma once

#include <hip/hip_runtime.h>

namespace nlo {

// A polynomial's coefficient, formed in scalar registers where it is used.
// FP64 instructions take no literal; left to itself the compiler keeps every
// coefficient of an unrolled loop in a pair of vector registers and spills
// them (the queue of the adaptive K1 rule: 192 bytes reloaded per node).
__host__ __device__ __forceinline__ double coef64(double k) {
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+s"(k));
#endif
    return k;
}

// 1 / b for |b| in [2^-1000, 2^1000]: Newton's iteration from the hardware
// estimate; the second step rounds (error below 1 ulp).
__device__ __forceinline__ double rcp64(double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    return fma(fma(-b, r, 1.0), r, r);
}

// a / b with 1 / b as above and a quotient that is an ordinary number; the
// residual a - b q corrects the rounding of a (1 / b).
__device__ __forceinline__ double div64(double a, double b) {
    double r = __builtin_amdgcn_rcp(b);
    r = fma(fma(-b, r, 1.0), r, r);
    const double q = a * r;
    return fma(fma(-b, q, a), r, q);
}

// 1 / sqrt(x) for ordinary x > 0: the hardware estimate (2^-24) and one step
// of third order.
__device__ __forceinline__ double rsqrt64(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(e, 0.375, 0.5), y);
}

// sqrt(x) for x = 0 and ordinary x > 0 (NaN below 0).
__device__ __forceinline__ double sqrt64(double x) {
    const double y = rsqrt64(x), g = x * y;
    const double r = fma(fma(-g, g, x), 0.5 * y, g);
    return x == 0.0 ? 0.0 : r;
}

// ln x for finite x > 0 (NaN for NaN).  x = 2^e (1 + f), 1 + f in [1/sqrt 2,
// sqrt 2); with s = f / (2 + f), ln(1 + f) = 2 atanh s = f - f^2/2 +
// s (f^2/2 + R(s^2)), where R(z) = 2 (z/3 + z^2/5 + ..) (degree 7,
// interpolated at Chebyshev nodes of z <= 0.0296, error 1.1e-17); f is exact.
// The reduction, the grouping of the terms and the two parts of ln 2 are those of
// FDLIBM's log (Sun Microsystems, 1993); the polynomial is its own.  What the
// two large terms e ln 2 + f and f^2/2 lose is added with the small ones.
__device__ __forceinline__ double log64(double x) {
    double m = __builtin_amdgcn_frexp_mant(x);  // [1/2, 1)
    int e = __builtin_amdgcn_frexp_exp(x);
    const int low = m < 0.70710678118654752440 ? 1 : 0;
    m = ldexp(m, low);
    e -= low;
    const double f = m - 1.0, d = m + 1.0;
    const double s = div64(f, d), z = s * s;
    double R = coef64(0.1462395660821188);
    R = fma(R, z, coef64(0.1533111258796017));
    R = fma(R, z, coef64(0.1818290749767122));
    R = fma(R, z, coef64(0.22222210881932927));
    R = fma(R, z, coef64(0.28571428627528794));
    R = fma(R, z, coef64(0.3999999999989607));
    R = fma(R, z, coef64(0.666666666666667));
    const double hf = 0.5 * f, h = hf * f, de = (double)e;
    // ln 2 = 0x1.62e42fee00000p-1 (33 bits: e times it is exact) + the rest
    const double low_part = fma(s, fma(R, z, h), de * 1.90821492927058770002e-10);
    const double b = fma(de, 6.93147180369123816490e-01, f);
    const double b_rest = fma(de, 6.93147180369123816490e-01, -b) + f;
    const double g = fma(-hf, f, b), g_rest = fma(-hf, f, b - g);
    return g + (low_part + (b_rest + g_rest));
}

// e^x for finite x (0 and infinity where it leaves the range, NaN for NaN):
// x = n ln 2 + r, |r| <= ln 2 / 2, e^r = 1 + r + r^2 P(r), P of degree 10
// interpolated at Chebyshev nodes (error 3e-19); the reduction as in FDLIBM's exp.
__device__ __forceinline__ double exp64(double x) {
    const double n = rint(x * 1.44269504088896340736);
    const double r = fma(-n, 1.90821492927058770002e-10, fma(-n, 6.93147180369123816490e-01, x));
    double p = coef64(2.0914686968086876e-09);
    p = fma(p, r, coef64(2.5105217004720745e-08));
    p = fma(p, r, coef64(2.75572736431103e-07));
    p = fma(p, r, coef64(2.7557255400206422e-06));
    p = fma(p, r, coef64(2.4801587325547743e-05));
    p = fma(p, r, coef64(0.00019841269874820627));
    p = fma(p, r, coef64(0.0013888888888883748));
    p = fma(p, r, coef64(0.008333333333326136));
    p = fma(p, r, coef64(0.04166666666666667));
    p = fma(p, r, coef64(0.1666666666666667));
    p = fma(p, r, coef64(0.5));
    const double v = 1.0 + r;
    return ldexp(v + fma(r * r, p, (1.0 - v) + r), (int)n);
}

// ln(1 + min(u, 1/u)) for u in [1e-18, 1e18]: 2 atanh w with w = u / (2 + u)
// or 1 / (1 + 2 u) (w <= 1/3), degree 10 in w^2 (error 7e-18 relative).
__device__ __forceinline__ double log1p_fold64(double u) {
    const bool big = u > 1.0;
    const double w = div64(big ? 1.0 : u, fma(big ? 2.0 : 1.0, u, big ? 1.0 : 2.0));
    const double z = w * w;
    double q = coef64(0.1616404561194353);
    q = fma(q, z, coef64(0.08800738486144674));
    q = fma(q, z, coef64(0.12001072809590713));
    q = fma(q, z, coef64(0.13314144209654935));
    q = fma(q, z, coef64(0.15385570064958623));
    q = fma(q, z, coef64(0.18181789436132859));
    q = fma(q, z, coef64(0.22222222717427864));
    q = fma(q, z, coef64(0.2857142856710876));
    q = fma(q, z, coef64(0.40000000000014585));
    q = fma(q, z, coef64(0.6666666666666666));
    return fma(w * z, q, w + w);
}

// sin^2 y for y in [0, pi]: with w = y (pi - y), sin y = cos((pi^2/4 -
// w)^1/2) is entire in w, and sin y / w is its degree-8 interpolant at
// Chebyshev nodes of [0, pi^2/4] (relative error 3e-20; all terms positive).
// pi is taken to twice the precision, so that the zero at pi keeps its place.
__device__ __forceinline__ double sin2_64(double y) {
    const double w = y * ((3.141592653589793116 - y) + 1.2246467991473532072e-16);
    double p = fma(w, coef64(1.5070686439285400088e-16), coef64(4.4416425756421120182e-14));
    p = fma(w, p, coef64(1.0560867829056239888e-11));
    p = fma(w, p, coef64(1.8975085675213420456e-9));
    p = fma(w, p, coef64(2.4609343506619309446e-7));
    p = fma(w, p, coef64(0.000021586579361110788302));
    p = fma(w, p, coef64(0.0011602715472401966982));
    p = fma(w, p, coef64(0.03225153443319948851));
    p = fma(w, p, coef64(0.31830988618379067155));
    const double s = w * p;
    return s * s;
}

}  // namespace nlo
