// Device-side BK physics: coupling, log-log splines held in LDS, the K1
// integrand and the K2 + Kf integrand in FP64 (reference formula) and FP32
// (cancellation-free formula).  Reference prefixes: S/ = torch_nlo_clean/src/
// nlo_torch/, K/ = S/custom_kernels/.
#pragma once

#include <hip/hip_runtime.h>

#include "bessel_j1_i1.hpp"
#include "fp64_math.hpp"
#include "common.hpp"

namespace nlo {

constexpr double kPi = 3.14159265358979323846;
constexpr double kLn2 = 0.69314718055994530942;
constexpr double kLog2e = 1.44269504088896340736;

// Physics constants derived once on the host from nlo_bk_physics.
struct BkConsts {
    double nc, nf, ksub, minr;
    double b0;          // (11 Nc - 2 Nf) / (12 pi)
    double log_mu0;     // 2 / 0.2 * ln 2.5
    double scale_num;   // 4 C2
    double lambda_qcd;
    double log_scale0;  // ln(4 C2 / Lambda^2)
    double norm;        // 1 / (8 pi^4)
    int symmetrize;
    int rc_lo, rc_nlo, resum_rc;  // NLO_RC_LO_*, NLO_RC_NLO_*, NLO_RESUM_RC_*
    int has_resum;      // Order resums the double logs (all but LO and NLO)
    int slog;           // ... and the single logs
    int fixed;          // every coupling is FIXED_AS (RC_LO or RC_NLO fixed)
    int thresholds;     // NF > 3: one-loop coupling with flavour thresholds
    int production;     // Balitsky LO, smallest resummation, DLOG_SLOG, smooth coupling
    double fixed_as;
    double log_4c2;     // ln(4 C2)
    double freeze;      // 2.5^2 Lambda^2 / (4 C2): the coupling freezes at d^2 = 1 / freeze
};

// -------------------------------------------------------------- coupling

// S/coupling.py:81-97: alpha = 1 / (b0 * 0.2 * logaddexp(2/0.2 ln 2.5,
// ln(4 C2 / (r^2 Lambda^2)) / 0.2)).
__device__ __forceinline__ double alpha_s64(double r, const BkConsts& c) {
    const double scale = c.scale_num / (r * r * c.lambda_qcd * c.lambda_qcd);
    const double right = log(scale) / 0.2;
    const double hi = fmax(c.log_mu0, right);
    return 1.0 / (c.b0 * (0.2 * (hi + log1p(exp(-fabs(c.log_mu0 - right))))));
}

// bk_alpha_s for NF > 3 (S/coupling.py:23-46): Nf and Lambda switched at
// 4 C2 / r^2 = 1.3^2 and 4.5^2, b0 = 11 - 2 Nf / 3, alpha = 4 pi / (b0 ln(4 C2 /
// (r^2 Lambda^2))), 1 where the logarithm's argument is below 1 or alpha > 1.
__device__ __forceinline__ double alpha_thresholds64(double r, const BkConsts& c) {
    const double dipolescale = c.scale_num / (r * r);
    double nf, lambda;
    if (dipolescale < 1.3 * 1.3) {
        nf = 3.0;
        lambda = 0.146159;
    } else if (dipolescale < 4.5 * 4.5) {
        nf = 4.0;
        lambda = 0.122944;
    } else {
        nf = 5.0;
        lambda = 0.0904389;
    }
    const double b0 = 11.0 - 2.0 * nf / 3.0;
    const double log_arg = c.scale_num / (r * r * (lambda * lambda));
    const double a = 4.0 * kPi / (b0 * log(log_arg));
    return (log_arg < 1.0 || a > 1.0) ? 1.0 : a;
}

// _alpha_s of S/bk_kernels/k1.py:158-169 and S/bk/derivatives.py:775-786:
// FIXED_AS, the smooth coupling (NF <= 3) or the threshold coupling.
__device__ __forceinline__ double alpha_any64(double r, const BkConsts& c) {
    if (c.fixed) return c.fixed_as;
    return c.thresholds ? alpha_thresholds64(r, c) : alpha_s64(r, c);
}

// The same threshold coupling from ln d (FP32 NLO integrand):
// ln(4 C2 / d^2) against 2 ln 1.3 and 2 ln 4.5, ln(arg) = that - 2 ln Lambda.
template <typename T>
__device__ __forceinline__ T alpha_thresholds_log(T log_d, T log_4c2) {
    const T lq = log_4c2 - T(2) * log_d;
    T nf = T(5), l2 = T(-4.806161588812351);  // 2 ln 0.0904389
    if (lq < T(0.5247285289349821)) {         // 2 ln 1.3
        nf = T(3);
        l2 = T(-3.8461204175059556);          // 2 ln 0.146159
    } else if (lq < T(3.0081547935525483)) {  // 2 ln 4.5
        nf = T(4);
        l2 = T(-4.192052623672091);           // 2 ln 0.122944
    }
    const T L = lq - l2;
    const T a = T(4.0 * kPi) / ((T(11) - T(2) * nf / T(3)) * L);
    return (L < T(0) || a > T(1)) ? T(1) : a;
}

// Coupling of the K2 + Kf integrand (_nlo_alpha_s, S/bk/derivatives.py:615-632):
// mode 0 = smooth coupling at the smallest distance (production), 1 = a
// constant per parent (FIXED_AS or alpha(r)), 2 = threshold coupling at the
// smallest distance.
template <typename T>
struct NloCoupling {
    int mode;
    T b0, log_mu0, log_scale0, log_4c2, as_const;
};

// ANYC = false: the production coupling (mode 0) compiled alone, so that the
// production kernels carry no code or registers of the other modes.
template <bool ANYC>
__device__ __forceinline__ double nlo_alpha_from_log(double log_min, const NloCoupling<double>& k) {
    if constexpr (ANYC) {
        if (k.mode == 1) return k.as_const;
        if (k.mode == 2) return alpha_thresholds_log<double>(log_min, k.log_4c2);
    }
    const double right = 5.0 * (k.log_scale0 - 2.0 * log_min);
    const double hi = fmax(k.log_mu0, right);
    return 1.0 / (k.b0 * (0.2 * (hi + log1p(exp(-fabs(k.log_mu0 - right))))));
}

// NloCoupling for a parent: the mode from the physics choice, the constant
// for FIXED_NLO / PARENT_NLO evaluated at r in FP64.
template <typename T>
__device__ __forceinline__ NloCoupling<T> nlo_coupling(double r, const BkConsts& c) {
    NloCoupling<T> k;
    k.b0 = (T)c.b0;
    k.log_mu0 = (T)c.log_mu0;
    k.log_scale0 = (T)c.log_scale0;
    k.log_4c2 = (T)c.log_4c2;
    k.as_const = T(0);
    if (c.fixed || c.rc_nlo == NLO_RC_NLO_FIXED) {
        k.mode = 1;
        k.as_const = (T)c.fixed_as;
    } else if (c.rc_nlo == NLO_RC_NLO_PARENT) {
        k.mode = 1;
        k.as_const = (T)alpha_any64(r, c);
    } else {
        k.mode = c.thresholds ? 2 : 0;
    }
    return k;
}

// Same coupling from ln r (FP32): right = 5 (ln(4 C2 / Lambda^2) - 2 ln r).
__device__ __forceinline__ float alpha_s32_log(float log_r, float b0, float log_mu0,
                                               float log_scale0) {
    const float right = 5.0f * (log_scale0 - 2.0f * log_r);
    const float hi = fmaxf(log_mu0, right);
    return 1.0f / (b0 * (0.2f * (hi + log1pf(expf(-fabsf(log_mu0 - right))))));
}

// --------------------------------------------------------------- splines

// A log-log spline staged in LDS: nodes x[n] = ln r_i and per-interval
// records {a, b, c, d} (structure of arrays would need four LDS reads).
template <typename T>
struct LdsSpline {
    const T* x;
    const T* rec;  // 4 (n - 1)
    int n;
    T x0, inv_h;   // ln r_0 and (n - 1) / (ln r_{n-1} - ln r_0)
    T log_min, log_max;
};

// searchsorted(x, v, right=True) - 1 clamped to [0, n - 2]
// (S/numerics/interpolation.py:55-56): the uniform-grid estimate, then exact
// correction against the nodes (one step on the log-uniform evolution grid).
template <typename T>
__device__ __forceinline__ int spline_interval(const LdsSpline<T>& s, T v) {
    int k = (int)((v - s.x0) * s.inv_h);
    k = k < 0 ? 0 : (k > s.n - 2 ? s.n - 2 : k);
    while (k > 0 && v < s.x[k]) --k;
    while (k < s.n - 2 && v >= s.x[k + 1]) ++k;
    return k;
}

template <typename T>
__device__ __forceinline__ T spline_poly(const LdsSpline<T>& s, T v) {
    const int k = spline_interval(s, v);
    const T dx = v - s.x[k];
    const T* c = s.rec + 4 * k;
    return c[0] + dx * (c[1] + dx * (c[2] + dx * c[3]));
}

// _evaluate_loglog (S/bk/derivatives.py:761-772) on a distance d.
__device__ __forceinline__ double loglog64(const LdsSpline<double>& s, double r_min, double r_max,
                                          double d, double underflow, double overflow) {
    const double ev = fmin(fmax(d, r_min), r_max);
    double out = exp(spline_poly(s, log(ev)));
    out = isfinite(out) ? out : 0.0;
    out = d < r_min ? underflow : out;
    return d > r_max ? overflow : out;
}

// Same from ln d: the clamp and the range tests done in log space.
template <typename T>
__device__ __forceinline__ T loglog_from_log(const LdsSpline<T>& s, T log_d, T underflow,
                                            T overflow) {
    const T lv = fmin(fmax(log_d, s.log_min), s.log_max);
    T out;
    if constexpr (sizeof(T) == 8)
        out = exp64(spline_poly(s, lv));
    else
        out = exp(spline_poly(s, lv));
    out = isfinite(out) ? out : T(0);
    out = log_d < s.log_min ? underflow : out;
    return log_d > s.log_max ? overflow : out;
}

// ------------------------------------------------------- K1 (FP64 only)

// Kernel_lo (S/bk_kernels/k1.py:20-155) for BALITSKY_LO, RESUM_RC_SMALLEST,
// NLO_RESUM_DLOG_SLOG, times the dipole of _lo_integrand
// (S/bk/derivatives.py:445-468), split so that everything that depends only
// on the daughter distance Y = z is computed once per z node (K1Z) and the
// theta loop evaluates the rest (k1_theta_term).  X^2 = (r - z)^2 +
// 4 r z sin^2(theta / 2) (the form K/bk/k1/kernel.cu:478-479 uses; it keeps
// X accurate near X -> 0).  Logarithms of distances are formed once and
// shared by the spline, the coupling and the resummation logs.

// alpha(d) from ln d (S/coupling.py:81-97): ln(4 C2 / (d^2 Lambda^2)) =
// log_scale0 - 2 ln d.  The denominator is returned too, so that ratios of
// couplings need no division: alpha_a / alpha_b = alpha_a * den_b.
// Far from the freezing scale (a factor above 1e18) the smooth-max term
// log1p(e^-|mu0 - right|) < 1e-18 is below half an ulp of hi >= mu0 = 10 ln 2.5, so
// hi + term rounds to hi: skipping it there changes no bit,
// and whole waves (small distances) skip them.
// e^(mu0 - right) is the fifth power of d^2 / (d^2 at the freezing), so the
// smooth-max term needs no exponential.
__device__ __forceinline__ double alpha_s64_den(double dsq, double log_d, const BkConsts& c) {
    const double right = (c.log_scale0 - 2.0 * log_d) * 5.0;  // / 0.2 within one rounding
    const double v = dsq * c.freeze, v2 = v * v, u = v2 * v2 * v;
    double sum = fmax(c.log_mu0, right);
    if (u > 1e-18 && u < 1e18) sum += log1p_fold64(u);
    return c.b0 * (0.2 * sum);
}

struct K1Parent {
    double r, log_r, n_r, a_r;
    double lo_coef;     // Nc / (2 pi^2) alpha(r)
    double fin_coef;    // alpha(r) Nc / (4 pi) (67/9 - pi^2/3 - 10/9 Nf/Nc)
    double log_ksub;
    double resum_on;    // 1 where r > 1.01 MINR (double-log resummation active)
    const double* j1tab;  // J1 Chebyshev pieces (LDS)
};

struct K1Z {
    double z, log_z, n_y, a_y, den_y, ly, inv_y2;
};

__device__ __forceinline__ double k1_theta_term(const K1Parent& P, const K1Z& Z, double s2,
                                                const LdsSpline<double>& sN, const BkConsts& c) {
    const double r = P.r, z = Z.z;
    const double xsq = (r - z) * (r - z) + 4.0 * r * z * s2;
    if (xsq < 1e-40 || z < 1e-20 || r < 1e-20) return 0.0;
    // X itself is never needed: ln X = ln(X^2) / 2, and squares compare alike
    const double lnX = 0.5 * log64(xsq), zsq = z * z;
    const double n_x = fmin(loglog_from_log(sN, lnX, 0.0, 1.0), 1.0);
    const double dipole = n_x + Z.n_y - P.n_r - n_x * Z.n_y;
    const double den_x = alpha_s64_den(xsq, lnX, c);
    // one division for both reciprocals: q = 1 / (den_x X^2)
    const double q = rcp64(den_x * xsq);
    const double a_x = q * xsq;
    const double inv_x2 = q * den_x;
    const double a_min = fmin(xsq, zsq) <= r * r ? (xsq <= zsq ? a_x : Z.a_y) : P.a_r;
    const double rxy2 = r * r * inv_x2 * Z.inv_y2;  // r^2 / (X^2 Y^2)
    // Kernel_lo: alpha_r (r^2/(X^2 Y^2) + (alpha_Y/alpha_X - 1)/Y^2 + (alpha_X/alpha_Y - 1)/X^2)
    double lo = P.lo_coef * (rxy2 + (Z.a_y * den_x - 1.0) * Z.inv_y2 + (a_x * Z.den_y - 1.0) * inv_x2);
    lo = isfinite(lo) ? lo : 0.0;
    const double xl = 4.0 * (lnX - P.log_r) * Z.ly;
    const double abar = a_min * (c.nc / kPi);  // loop-invariant quotient
    // J1(2a)/a (xl >= 0) or I1(2a)/a (xl < 0), a^2 = abar |xl| (k1.py:108-132):
    // one series in s = -abar xl for |s| <= 16 (no divergence between the two
    // sides), the J1 table or the large-argument I1 beyond
    const double sres = -abar * xl;
    double dlog = 1.0;
    if (P.resum_on != 0.0 && sres != 0.0) {
        if (fabs(sres) <= 16.0) {
            dlog = j1_i1_series(sres);
        } else {
            const double as_x = sqrt(fabs(sres));
            dlog = sres < 0.0 ? j1_over_half_x(2.0 * as_x, P.j1tab) : i1_over_half_x(2.0 * as_x);
        }
    }
    if (!isfinite(dlog)) return 0.0;
    // ln(KSUB r^2 / min(X, Y)^2): the single-log exponent of both slog terms
    const double lmin = xsq <= zsq ? lnX : Z.log_z;
    const double slog_exp = -abar * (11.0 / 12.0) * fabs(P.log_ksub + 2.0 * (P.log_r - lmin));
    const double slog = exp64(slog_exp);
    const double lo_single = P.lo_coef * rxy2;
    const double k1fin = lo * P.fin_coef;
    return (dlog * slog * lo - lo_single * slog_exp + k1fin) * dipole;
}

// ------------------------------------------ K1 for every physics choice

// Kernel_lo (S/bk_kernels/k1.py:20-155) for any RC_LO / RESUM_RC / Order
// choice, at valid distances X, Y (logs given).  j1tab: the J1 table in LDS.
__device__ inline double kernel_lo_any(double r, double log_r, double X, double lnX, double Y,
                                       double lnY, const BkConsts& c, const double* j1tab) {
    const double mn = fmin(fmin(X, Y), r);
    const double a_r = alpha_any64(r, c);
    const double rxy2 = (r / (X * Y)) * (r / (X * Y));
    const double pref = c.nc / (2.0 * kPi * kPi);
    double lo, a_scale;
    switch (c.rc_lo) {
        case NLO_RC_LO_SMALLEST:
            a_scale = alpha_any64(mn, c);
            lo = pref * a_scale * rxy2;
            break;
        case NLO_RC_LO_PARENT:
            a_scale = a_r;
            lo = pref * a_r * rxy2;
            break;
        case NLO_RC_LO_FAC: {
            const double ab_r = a_r * c.nc / kPi;
            const double ab_x = alpha_any64(X, c) * c.nc / kPi;
            const double ab_y = alpha_any64(Y, c) * c.nc / kPi;
            a_scale = a_r;
            lo = 1.0 / (2.0 * kPi) /
                 (1.0 / ab_r + (X * X - Y * Y) / (r * r) * (ab_x - ab_y) / (ab_x * ab_y)) * rxy2;
            break;
        }
        case NLO_RC_LO_BEUF: {
            const double reff2 = r * r * pow(Y * Y / (X * X), (X * X - Y * Y) / (r * r));
            a_scale = alpha_any64(sqrt(reff2), c);
            const double q = r / (X * Y + 1e-40);
            lo = pref * a_scale * q * q;
            break;
        }
        default: {  // BALITSKY_LO, FIXED_LO
            const double a_x = alpha_any64(X, c), a_y = alpha_any64(Y, c);
            a_scale = a_r;
            lo = pref * a_r * (rxy2 + (a_y / a_x - 1.0) / (Y * Y) + (a_x / a_y - 1.0) / (X * X));
            break;
        }
    }
    lo = isfinite(lo) ? lo : 0.0;
    if (!c.has_resum) return lo;
    const double a_res = c.resum_rc == NLO_RESUM_RC_PARENT  ? a_r
                         : c.resum_rc == NLO_RESUM_RC_FIXED ? c.fixed_as
                                                            : alpha_any64(mn, c);
    const double abar = a_res * c.nc / kPi;
    const double xl = 4.0 * (lnX - log_r) * (lnY - log_r);
    const double sres = -abar * xl;  // a^2 with the J1 side negative, as in k1_theta_term
    double dlog = 1.0;
    if (r > 1.01 * c.minr && sres != 0.0) {
        if (fabs(sres) <= 16.0) {
            dlog = j1_i1_series(sres);
        } else {
            const double as_x = sqrt(fabs(sres));
            dlog = sres < 0.0 ? j1_over_half_x(2.0 * as_x, j1tab) : i1_over_half_x(2.0 * as_x);
        }
    }
    if (!isfinite(dlog)) return 0.0;
    double slog = 1.0, slog_exp = 0.0;
    if (c.slog) {
        // ln(KSUB r^2 / min(X, Y)^2), shared by both single-log terms
        slog_exp = -abar * (11.0 / 12.0) * fabs(log(c.ksub) + 2.0 * (log_r - fmin(lnX, lnY)));
        slog = exp(slog_exp);
    }
    const double lo_single = pref * a_scale * rxy2;
    const double fin = a_scale * c.nc / (4.0 * kPi) * (67.0 / 9.0 - kPi * kPi / 3.0 - 10.0 / 9.0 * c.nf / c.nc);
    return dlog * slog * lo - lo_single * slog_exp + lo * fin;
}

// Amplitude history for the kinematical constraint: rows N(r_grid, y_k),
// k < *rows, in HBM; the current rapidity is the last row's.
struct K1History {
    const double* y;
    const double* N;
    const double* r;
    const int32_t* rows;  // device row count, read by the kernel (clamped to capacity)
    int n;
    int capacity;
};

// NaturalCubicSpline on six nodes evaluated at v (S/numerics/interpolation.py:10-68).
__device__ inline double natural6(const double* x, const double* y, double v) {
    double h[5], up[4], sol[4];
    for (int i = 0; i < 5; ++i) h[i] = x[i + 1] - x[i];
    for (int i = 0; i < 4; ++i) {
        const double diag = 2.0 * (h[i] + h[i + 1]);
        const double rhs = 6.0 * ((y[i + 2] - y[i + 1]) / h[i + 1] - (y[i + 1] - y[i]) / h[i]);
        const double den = i == 0 ? diag : diag - h[i] * up[i - 1];
        up[i] = h[i + 1] / den;
        sol[i] = (rhs - (i == 0 ? 0.0 : h[i] * sol[i - 1])) / den;
    }
    for (int i = 2; i >= 0; --i) sol[i] -= up[i] * sol[i + 1];
    int k = 0;
    while (k < 4 && x[k + 1] <= v) ++k;
    const double m0 = k == 0 ? 0.0 : sol[k - 1], m1 = k == 4 ? 0.0 : sol[k];
    const double b = (y[k + 1] - y[k]) / h[k] - h[k] * (2.0 * m0 + m1) / 6.0;
    const double dx = v - x[k];
    return y[k] + dx * (b + dx * (m0 / 2.0 + dx * (m1 - m0) / (6.0 * h[k])));
}

// _interpolate_history_N (S/bk/derivatives.py:712-758) at (d, rapidity),
// 0 <= rapidity <= the last row's rapidity; the last row is read through the
// current spline sN.
__device__ inline double history_n(double d, double log_d, double rapidity, const K1History& H,
                                   int rows, const LdsSpline<double>& sN) {
    int lo = 0, hi = rows;  // first row with y > rapidity
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (H.y[mid] <= rapidity) lo = mid + 1; else hi = mid;
    }
    const int yind = lo - 1 < 0 ? 0 : lo - 1;
    double out;
    if (yind == rows - 1) {
        out = loglog_from_log(sN, log_d, 0.0, 1.0);
    } else {
        int a = 0, b = H.n;  // first node with r > d
        while (a < b) {
            const int mid = (a + b) >> 1;
            if (H.r[mid] <= d) a = mid + 1; else b = mid;
        }
        const int rind = a - 1;
        const int start = rind - 3 > 0 ? rind - 3 : 0;
        if (start + 6 > H.n) {
            out = 1.0;
        } else {
            double x[6], yl[6], yu[6];
            for (int i = 0; i < 6; ++i) {
                x[i] = H.r[start + i];
                yl[i] = H.N[(size_t)yind * H.n + start + i];
                yu[i] = H.N[(size_t)(yind + 1) * H.n + start + i];
            }
            double v = d;
            if (v < x[0]) v = x[0] * 1.00001;
            if (v > x[5]) v = x[5] * 0.999999;
            const double nl = natural6(x, yl, v), nu = natural6(x, yu, v);
            const double frac = (rapidity - H.y[yind]) / (H.y[yind + 1] - H.y[yind]);
            out = nl + frac * (nu - nl);
        }
    }
    return fmin(fmax(out, 0.0), 1.0);
}

// The K1 integrand (_lo_integrand, S/bk/derivatives.py:434-468) for any
// physics choice, with the kinematical constraint when H.rows is set.
__device__ inline double k1_theta_term_any(const K1Parent& P, const K1Z& Z, double s2,
                                           const LdsSpline<double>& sN, const BkConsts& c,
                                           const K1History& H, int rows, double rapidity) {
    const double r = P.r, z = Z.z;
    const double xsq = (r - z) * (r - z) + 4.0 * r * z * s2;
    if (xsq < 1e-40 || z < 1e-20 || r < 1e-20) return 0.0;
    const double X = sqrt(xsq);
    const double lnX = log(X);
    const double k = kernel_lo_any(r, P.log_r, X, lnX, z, Z.log_z, c, P.j1tab);
    if (rows == 0) {
        const double n_x = fmin(loglog_from_log(sN, lnX, 0.0, 1.0), 1.0);
        return k * (n_x + Z.n_y - P.n_r - n_x * Z.n_y);
    }
    // rapidity shifted by max(0, ln(min(X, Y)^2 / r^2)); cut below zero
    const double delta = fmax(2.0 * (fmin(lnX, Z.log_z) - P.log_r), 0.0);
    const double shifted = rapidity - delta;
    if (shifted < 0.0) return 0.0;
    const double s02 = 1.0 - history_n(X, lnX, shifted, H, rows, sN);
    const double s12 = 1.0 - history_n(z, Z.log_z, shifted, H, rows, sN);
    return k * (-s02 * s12 + (1.0 - P.n_r));
}

// -------------------------------------------------- K2 + Kf, FP64 direct

struct NloValue64 {
    double total, k2, kf;
};

// One order of the kernels (S/bk_kernels/k2.py:24-36, kf.py:28-38) from a2 =
// X^2 z'^2, b2 = X'^2 z^2, d = a2 - b2 and ratio = X z' / (X' z); the other
// order has a2 and b2, the sign of d and the ratio inverted.
struct NloKernels64 {
    double k2, kf;
};

__device__ __forceinline__ NloKernels64 nlo_kernels64(double a2, double b2, double d, double ratio, double rsq,
                                                      double zsq, double iz, double nf_over_nc) {
    const double L = 2.0 * log64(ratio), t = L * rcp64(d), rz = rsq * zsq, iz4 = iz * iz;
    NloKernels64 k;
    k.k2 = ((a2 + b2 - 4.0 * rz) * t - 2.0) * iz4 + rcp64(a2) * (rsq * rsq * t + rsq * iz * L);
    k.kf = (2.0 - (a2 + b2 - rz) * t) * iz4 * nf_over_nc;
    k.k2 = isfinite(k.k2) ? k.k2 : 0.0;  // d = 0, and beyond the range
    k.kf = isfinite(k.kf) ? k.kf : 0.0;
    return k;
}

// The same two kernels with every quotient and function of the library, one
// order at a time, for the passes that refine the grids.
__device__ __forceinline__ double kernel_nlo64(double r, double X, double Y, double X2, double Y2, double Z,
                                               double z4) {
    const double a2 = (X * Y2) * (X * Y2), b2 = (X2 * Y) * (X2 * Y);
    const double diff = a2 - b2;
    const double rz = r * Z;
    const double k = -2.0 / z4 + ((a2 + b2 - 4.0 * rz * rz) / (z4 * diff) + (r * r) * (r * r) / (a2 * diff) +
                                  r * r / ((X * Y2 * Z) * (X * Y2 * Z))) *
                                     2.0 * log(X * Y2 / (X2 * Y));
    return isfinite(k) ? k : 0.0;
}

__device__ __forceinline__ double kernel_nlo_fermion64(double r, double X, double Y, double X2, double Y2, double Z,
                                                       double z4, double nf, double nc) {
    const double a2 = (X * Y2) * (X * Y2), b2 = (X2 * Y) * (X2 * Y);
    const double rz = r * Z;
    double k = 2.0 / z4 - (a2 + b2 - rz * rz) / (z4 * (a2 - b2)) * 2.0 * log(X * Y2 / (X2 * Y));
    k = k * nf / nc;
    return isfinite(k) ? k : 0.0;
}

// |e^(lz) - r e^(i t)|^2, s = sin(t / 2).
__device__ __forceinline__ double nlo_distance_sq64(double r, double z, double s) {
    const double d = r - z;
    return fma(d, d, 4.0 * r * z * s * s);
}

// _nlo_integrand (S/bk/derivatives.py:521-612) times exp(2 ln z + 2 ln z')
// (S/bk/derivatives.py:335), with the reference's kernels and S dipoles.
//
// Bound by FP64 issue.  The distances keep the library's exponential and sine
// and the kernels' cancelling parts the formula's own steps;
// splines, coupling and scale, which nothing amplifies, take one logarithm per
// squared distance, and the quotients shared reciprocals.  RK2 step of 2^18
// points on 256 nodes 6.31 -> 4.40 ms; the sums keep the values of the plain
// evaluation to 1.2e-11 in 210 steps.  (Squared distances throughout, with one
// logarithm for both orders of the kernels, took 3.45 ms, but left them by 6e-8.)
//
// PLAIN (the passes with a histogram): every step by the library.  An edge that
// moves by an ulp draws other roundings from the cancelling samples of all
// passes behind it, so the grids have to come out to the last bit: with the
// shared logarithms in those passes too, 5 of 150 FP64 evolutions were off by
// more than 1e-10, up to 5e-8.
template <bool ANYC, bool PLAIN>
__device__ NloValue64 nlo_integrand64(double r, double log_r, double lz, double lz2, double tz, double tz2,
                                      const LdsSpline<double>& sS, double r_min, double r_max, const BkConsts& c) {
    NloValue64 out{0.0, 0.0, 0.0};
    const double z = exp(lz), z2 = exp(lz2);
    const double xsq = nlo_distance_sq64(r, z, sin(tz / 2.0));
    const double x2sq = nlo_distance_sq64(r, z2, sin(tz2 / 2.0));
    const double zsq = nlo_distance_sq64(z, z2, sin((tz - tz2) / 2.0));
    if (xsq < 1e-40 || z < 1e-20 || x2sq < 1e-40 || z2 < 1e-20 || zsq < 1e-40) return out;
    double S_X, S_Y, S_X2, S_Y2, S_Z, as, k, ks, kf, kfs, jac;
    // _nlo_alpha_s (S/bk/derivatives.py:615-632)
    const bool any_fixed = c.fixed || c.rc_nlo == NLO_RC_NLO_FIXED;
    if constexpr (PLAIN) {
        const double X = sqrt(xsq), X2 = sqrt(x2sq), Z = sqrt(zsq), z4 = Z * Z * Z * Z;
        S_X = loglog64(sS, r_min, r_max, X, 1.0, 0.0);
        S_Y = loglog64(sS, r_min, r_max, z, 1.0, 0.0);
        S_X2 = loglog64(sS, r_min, r_max, X2, 1.0, 0.0);
        S_Y2 = loglog64(sS, r_min, r_max, z2, 1.0, 0.0);
        S_Z = loglog64(sS, r_min, r_max, Z, 1.0, 0.0);
        const double dmin = fmin(fmin(fmin(r, X), z), fmin(fmin(X2, z2), Z));
        if constexpr (ANYC)
            as = any_fixed ? c.fixed_as : alpha_any64(c.rc_nlo == NLO_RC_NLO_PARENT ? r : dmin, c);
        else
            as = alpha_s64(dmin, c);
        k = kernel_nlo64(r, X, z, X2, z2, Z, z4);
        ks = kernel_nlo64(r, X2, z2, X, z, Z, z4);
        kf = kernel_nlo_fermion64(r, X, z, X2, z2, Z, z4, c.nf, c.nc);
        kfs = kernel_nlo_fermion64(r, X2, z2, X, z, Z, z4, c.nf, c.nc);
        jac = exp(2.0 * lz + 2.0 * lz2);
    } else {
        const double X = sqrt64(xsq), X2 = sqrt64(x2sq);
        const double lx = 0.5 * log64(xsq), lx2 = 0.5 * log64(x2sq), lZ = 0.5 * log64(zsq);
        S_X = loglog_from_log(sS, lx, 1.0, 0.0);
        S_Y = loglog_from_log(sS, lz, 1.0, 0.0);
        S_X2 = loglog_from_log(sS, lx2, 1.0, 0.0);
        S_Y2 = loglog_from_log(sS, lz2, 1.0, 0.0);
        S_Z = loglog_from_log(sS, lZ, 1.0, 0.0);
        const double rsq = r * r;
        const double dminsq = fmin(fmin(fmin(rsq, xsq), z * z), fmin(fmin(x2sq, z2 * z2), zsq));
        if constexpr (ANYC) {
            as = any_fixed ? c.fixed_as : alpha_any64(c.rc_nlo == NLO_RC_NLO_PARENT ? r : sqrt(dminsq), c);
        } else {
            const double lmin = fmin(fmin(fmin(log_r, lx), lz), fmin(fmin(lx2, lz2), lZ));
            as = rcp64(alpha_s64_den(dminsq, lmin, c));
        }
        const double iz = rcp64(zsq);
        // p ~ q: the rounding of p, q, their squares and quotients is amplified by
        // 1 / d, so that another order of these steps would move a sum by up to 6e-8
        const double p = X * z2, q = X2 * z, a2 = p * p, b2 = q * q, d = fma(-q, q, a2);
        const double nf_over_nc = c.nf / c.nc;
        const NloKernels64 ka = nlo_kernels64(a2, b2, d, div64(p, q), rsq, zsq, iz, nf_over_nc);
        const NloKernels64 kb = nlo_kernels64(b2, a2, -d, div64(q, p), rsq, zsq, iz, nf_over_nc);
        k = ka.k2, ks = kb.k2, kf = ka.kf, kfs = kb.kf;
        const double zz = z * z2;
        jac = zz * zz;
    }
    double dip = -(S_X * S_Z * S_Y2 - S_X * S_Y);
    double dips = -(S_X2 * S_Z * S_Y - S_X2 * S_Y2);
    if (fabs(k) > 1e10 && fabs(dip) < 1e-10) { k = 0.0; dip = 0.0; }
    if (fabs(ks) > 1e10 && fabs(dips) < 1e-10) { ks = 0.0; dips = 0.0; }
    double k2r = c.symmetrize ? (k * dip + ks * dips) / 2.0 : k * dip;
    double kfr = 0.0;
    if (c.nf > 0.0) {
        const double df = S_Y * (S_X2 - S_X);
        const double dfs = S_Y2 * (S_X - S_X2);
        kfr = -(c.symmetrize ? (kf * df + kfs * dfs) / 2.0 : kf * df);
    }
    const double scale = (as * c.nc) * (as * c.nc) * c.norm * jac;
    k2r *= scale;
    kfr *= scale;
    out.k2 = isfinite(k2r) ? k2r : 0.0;
    out.kf = isfinite(kfr) ? kfr : 0.0;
    out.total = out.k2 + out.kf;
    return out;
}

// ------------------------------------- K2 + Kf, cancellation-free kernels

// g(L) = L coth L - 1 (even).  |L| < 1: L^2 P(L^2) / Q(L^2) with
// L cosh L - sinh L = L^3 P(L^2), sinh L = L Q(L^2), both series positive;
// otherwise |L| + h(|L|) - 1.
template <typename T>
__device__ __forceinline__ T coth_minus_one(T L);

template <>
__device__ __forceinline__ double coth_minus_one<double>(double L) {
    L = fabs(L);
    if (L < 1.0) {
        const double y = L * L;
        const double p =
            ((((((((((1.0 / 1175091669949317120000.0) * y + 1.0 / 2554547108585472000.0) * y +
                    1.0 / 6758061133824000.0) * y + 1.0 / 22230464256000.0) * y +
                  1.0 / 93405312000.0) * y + 1.0 / 518918400.0) * y + 1.0 / 3991680.0) * y +
               1.0 / 45360.0) * y + 1.0 / 840.0) * y + 1.0 / 30.0) * y + 1.0 / 3.0;
        const double q =
            (((((((((((1.0 / 25852016738884976640000.0) * y + 1.0 / 51090942171709440000.0) * y +
                     1.0 / 121645100408832000.0) * y + 1.0 / 355687428096000.0) * y +
                   1.0 / 1307674368000.0) * y + 1.0 / 6227020800.0) * y + 1.0 / 39916800.0) * y +
                1.0 / 362880.0) * y + 1.0 / 5040.0) * y + 1.0 / 120.0) * y + 1.0 / 6.0) * y + 1.0;
        return y * p / q;
    }
    return L + 2.0 * L / expm1(2.0 * L) - 1.0;
}

template <>
__device__ __forceinline__ float coth_minus_one<float>(float L) {
    L = fabsf(L);
    if (L < 1.0f) {
        const float y = L * L;
        const float p = ((((1.0f / 518918400.0f) * y + 1.0f / 3991680.0f) * y + 1.0f / 45360.0f) * y +
                         1.0f / 840.0f) * y + 1.0f / 30.0f;
        const float q = ((((1.0f / 39916800.0f) * y + 1.0f / 362880.0f) * y + 1.0f / 5040.0f) * y +
                         1.0f / 120.0f) * y + 1.0f / 6.0f;
        return y * (p * y + 1.0f / 3.0f) / (q * y + 1.0f);
    }
    return L + 2.0f * L / expm1f(2.0f * L) - 1.0f;
}

// ln(X / Y) with X^2 = (r - z)^2 + 4 r z sin^2(theta / 2), Y = z:
// (X^2 - z^2) / z^2 = rho (rho - 2 cos theta), rho = r / z.
template <typename T>
__device__ __forceinline__ T log_x_over_y(T r, T z, T log_z, T cos_t, T xsq);

template <>
__device__ __forceinline__ double log_x_over_y<double>(double r, double z, double log_z,
                                                       double cos_t, double xsq) {
    const double rho = r / z;
    const double u = rho * (rho - 2.0 * cos_t);
    return fabs(u) < 0.5 ? 0.5 * log1p(u) : 0.5 * log(xsq) - log_z;
}

template <>
__device__ __forceinline__ float log_x_over_y<float>(float r, float z, float log_z, float cos_t,
                                                     float xsq) {
    const float rho = r / z;
    const float u = rho * (rho - 2.0f * cos_t);
    return fabsf(u) < 0.5f ? 0.5f * log1pf(u) : 0.5f * logf(xsq) - log_z;
}

struct NloValue32 {
    float total, k2, kf;
};

// The K2 + Kf integrand of S/bk/derivatives.py:521-612 with the kernels in
// cancellation-free form (multiplied by J = z^2 z'^2):
//   K2 J  = 2 A^2 g - 4 h B^2 + h C^2 + 2 L D^2
//   K2s J = 2 A^2 g - 4 h' D^2 + h' C^2 - 2 L B^2
//   Kf J  = (-2 A^2 g + h B^2) Nf / Nc,  Kfs J = (-2 A^2 g + h' D^2) Nf / Nc
// L = ln(X Y' / (X' Y)), g = L coth L - 1, h = 2L / (e^{2L} - 1),
// h' = h e^{2L}, A = z z' / Z^2, B = r z' / (X' Z), C = r^2 / (X X'),
// D = r z / (X Z); dipoles in N = 1 - S form.  Every quantity is a ratio of
// distances, so FP32 neither overflows nor cancels; no FP64 band is needed.
template <typename T>
struct NloStable {
    T total, k2, kf;
};

template <typename T, bool ANYC>
__device__ __forceinline__ NloStable<T> nlo_integrand_stable(T r, T log_r, T lz, T lz2, T tz, T tz2,
                                                             const LdsSpline<T>& sN,
                                                             const NloCoupling<T>& cpl, T nf_over_nc,
                                                             T nc, T norm, bool symmetrize) {
    NloStable<T> out{T(0), T(0), T(0)};
    const T z = exp(lz), z2 = exp(lz2);
    const T c1 = cos(tz), c2 = cos(tz2);
    const T s1 = sin(T(0.5) * tz), s2 = sin(T(0.5) * tz2), s3 = sin(T(0.5) * (tz - tz2));
    const T xsq = (r - z) * (r - z) + T(4) * r * z * s1 * s1;
    const T x2sq = (r - z2) * (r - z2) + T(4) * r * z2 * s2 * s2;
    const T zsq = (z - z2) * (z - z2) + T(4) * z * z2 * s3 * s3;
    const T tiny = sizeof(T) == 4 ? T(1e-37) : T(1e-40);
    if (!(xsq >= tiny) || !(x2sq >= tiny) || !(zsq >= tiny)) return out;
    const T X = sqrt(xsq), X2 = sqrt(x2sq), Z = sqrt(zsq);
    const T lxy = log_x_over_y<T>(r, z, lz, c1, xsq);
    const T lx2y2 = log_x_over_y<T>(r, z2, lz2, c2, x2sq);
    const T log_x = lz + lxy, log_x2 = lz2 + lx2y2, log_zz = T(0.5) * log(zsq);
    // N at the five distances: r_min..r_max, N -> 0 below and 1 above.
    const T n_x = loglog_from_log(sN, log_x, T(0), T(1));
    const T n_y = loglog_from_log(sN, lz, T(0), T(1));
    const T n_x2 = loglog_from_log(sN, log_x2, T(0), T(1));
    const T n_y2 = loglog_from_log(sN, lz2, T(0), T(1));
    const T n_z = loglog_from_log(sN, log_zz, T(0), T(1));
    const T sx = T(1) - n_x, sx2 = T(1) - n_x2;
    T dip = sx * (n_z + n_y2 - n_y - n_z * n_y2);
    T dips = sx2 * (n_z + n_y - n_y2 - n_z * n_y);

    const T L = lxy - lx2y2;
    const T g = coth_minus_one<T>(L);
    const T e2l = exp(T(2) * L);
    const T h = L == T(0) ? T(1) : T(2) * L / expm1(T(2) * L);
    const T hm = h * e2l;
    const T A = z * z2 / zsq, B = r * z2 / (X2 * Z), C = r * r / (X * X2), D = r * z / (X * Z);
    const T A2g = T(2) * A * A * g;
    T k = A2g - T(4) * h * B * B + h * C * C + T(2) * L * D * D;
    T ks = A2g - T(4) * hm * D * D + hm * C * C - T(2) * L * B * B;
    // cut of S/bk/derivatives.py:589-594: |K2| > 1e10 with |dipole| < 1e-10
    const T cut = T(1e10) * exp(T(2) * (lz + lz2));
    if (fabs(k) > cut && fabs(dip) < T(1e-10)) { k = T(0); dip = T(0); }
    if (fabs(ks) > cut && fabs(dips) < T(1e-10)) { ks = T(0); dips = T(0); }
    T k2r = symmetrize ? (k * dip + ks * dips) * T(0.5) : k * dip;
    T kfr = T(0);
    if (nf_over_nc > T(0)) {
        const T kf = (-A2g + h * B * B) * nf_over_nc;
        const T kfs = (-A2g + hm * D * D) * nf_over_nc;
        const T df = (T(1) - n_y) * (n_x - n_x2);
        const T dfs = (T(1) - n_y2) * (n_x2 - n_x);
        kfr = -(symmetrize ? (kf * df + kfs * dfs) * T(0.5) : kf * df);
    }
    const T log_min = fmin(fmin(fmin(log_r, log_x), lz), fmin(fmin(log_x2, lz2), log_zz));
    const T as = nlo_alpha_from_log<ANYC>(log_min, cpl);
    const T scale = (as * nc) * (as * nc) * norm;
    k2r *= scale;
    kfr *= scale;
    out.k2 = isfinite(k2r) ? k2r : T(0);
    out.kf = isfinite(kfr) ? kfr : T(0);
    out.total = out.k2 + out.kf;
    return out;
}

// ------------------------------------------- FP32 path: fast primitives
//
// The FP32 integrand works in units of the parent size r and in base-2
// logarithms: the VEGAS map hands it t = log2(z / r) (its bin table holds the
// logarithms relative to log2 r, formed in FP64), so every logarithm of a
// distance comes from the hardware log2 with no conversion, and near z = r,
// where the largest samples sit, t is small and carries its full relative
// precision (log2 z of a small distance would round z by up to 1e-6).

constexpr float kLn2f = 0.693147182f;
constexpr float kLog2ef = 1.44269502f;

__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float flog2(float x) { return __builtin_amdgcn_logf(x); }

__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }

__device__ __forceinline__ float frsq(float x) { return __builtin_amdgcn_rsqf(x); }

// Least and largest values, none of them a signalling NaN: the library forms
// canonicalise every operand that reaches a loop from outside by a v_max.
__device__ __forceinline__ float fmin3(float a, float b, float c) {
    float o;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(o) : "v"(a), "v"(b), "v"(c));
    return o;
}
__device__ __forceinline__ float fmax3(float a, float b, float c) {
    float o;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(o) : "v"(a), "v"(b), "v"(c));
    return o;
}
__device__ __forceinline__ float fmax2(float a, float b) {
    float o;
    asm("v_max_f32 %0, %1, %2" : "=v"(o) : "v"(a), "v"(b));
    return o;
}
// Keeps what follows inside its branch (the compiler would run it always and
// select, which costs every wave).
__device__ __forceinline__ void keep_branch(float& v) { asm volatile("" : "+v"(v)); }

// 4 sin^2 y from w = |y| (pi - |y|), 0 <= w <= pi^2/4: |sin y| = cos((pi^2/4 -
// w)^1/2) is entire in w, and 2 |sin y| / w is its degree-4 interpolant at
// Chebyshev nodes of that range (relative error 1e-9; all terms positive), so
// that no fold into [0, pi/2] is needed.
__device__ __forceinline__ float f4sin2_from(float w) {
    float p = fmaf(w, 5.161262147e-07f, 4.312110734e-05f);
    p = fmaf(w, p, 2.320589108e-03f);
    p = fmaf(w, p, 6.450305465e-02f);
    p = fmaf(w, p, 6.366197731e-01f);
    const float s = w * p;
    return s * s;
}

// |y| <= pi.  pi - |y| is exact near pi, with the low part of pi added.  pi:
// 3.14159274f in a vector register.
__device__ __forceinline__ float f4sin2(float y, float pi) {
    return f4sin2_from(fabsf(y) * ((pi - fabsf(y)) + -8.74227766e-8f));
}

// |y| <= 2 pi: the difference of two half-angles leaves [-pi, pi] where one of
// them lies in a bin across pi/2 and the grids of the two differ.  With u = pi -
// |y|, sin^2 y = sin^2 u and w = |u| (pi - |u|); outside [-pi, pi] the polynomial
// is off by 4e-8 at 1.03 pi, 6e-5 at 1.3 pi and 1e-3 at 1.5 pi.
__device__ __forceinline__ float f4sin2_wide(float y, float pi) {
    const float u = (pi - fabsf(y)) + -8.74227766e-8f;
    return f4sin2_from(fabsf(u) * fminf(fabsf(y), 6.28318548f - fabsf(y)));
}

// log2(1 + u) / 2 for |u| < 0.5: atanh(s) log2(e) with s = u / (2 + u),
// |s| < 0.2, the series to s^9 with log2(e) folded into its coefficients.
__device__ __forceinline__ float fhalf_log2_1p_small(float u) {
    const float s = u * frcp(2.0f + u);
    const float s2 = s * s;
    float p = fmaf(s2, 0.160299450f, 0.206099287f);  // log2(e) / 9, / 7
    p = fmaf(s2, p, 0.288539022f);                  // log2(e) / 5
    p = fmaf(s2, p, 0.480898350f);                  // log2(e) / 3
    p = fmaf(s2, p, 1.44269502f);                   // log2(e)
    return s * p;
}

// 2^t - 1 for |t ln 2| < 1/4: sum_k (ln 2)^k t^k / k!, k = 1..6 (relative error
// < 2e-8).
__device__ __forceinline__ float fexp2m1_small(float t) {
    float p = fmaf(t, 1.54035304e-4f, 1.33335581e-3f);  // (ln 2)^6 / 720, (ln 2)^5 / 120
    p = fmaf(t, p, 9.61812911e-3f);                     // (ln 2)^4 / 24
    p = fmaf(t, p, 5.55041087e-2f);                     // (ln 2)^3 / 6
    p = fmaf(t, p, 2.40226507e-1f);                     // (ln 2)^2 / 2
    p = fmaf(t, p, 6.93147181e-1f);                     // ln 2
    return t * p;
}

// h(L) = 2L / (e^{2L} - 1), h(-L) = h(L) e^{2L} and g(L) = L coth L - 1 =
// h(|L|) + |L| - 1 for x = 2L given also in base 2 (x2 = 2L log2 e, so e^{2L} =
// 2^x2 with no rounding of the argument).  |x| < 0.25: the Bernoulli series g =
// x^2/12 - x^4/720 + x^6/30240, h = g + 1 - x/2; else h from e^{2L} (no
// cancellation there; the second form avoids 1 - e^x for x << 0; x2 is
// clamped at 124, e^86), and g by its seven-term series in y = L^2 for |L| < 1
// (sum_n 2^2n B_2n L^2n / (2n)!, whose terms fall by ~1/pi^2).
__device__ __forceinline__ void fhg(float x, float x2, float& h, float& hm, float& g) {
    if (fabsf(x) < 0.25f) {
        const float xx = x * x;
        float p = fmaf(xx, 1.0f / 30240.0f, -1.0f / 720.0f);
        p = fmaf(xx, p, 1.0f / 12.0f);
        g = xx * p;
        h = g + fmaf(x, -0.5f, 1.0f);
        hm = h + x;
    } else {
        const float E = fexp2(fminf(x2, 124.0f));
        h = x * frcp(E - 1.0f);
        hm = h * E;
        const float aL = fabsf(0.5f * x);
        if (aL < 1.0f) {
            const float y = aL * aL;
            float p = fmaf(y, 2.19259479e-7f, -2.16440428e-6f);
            p = fmaf(y, p, 2.13777992e-5f);
            p = fmaf(y, p, -2.11640212e-4f);
            p = fmaf(y, p, 2.11640212e-3f);
            p = fmaf(y, p, -2.22222222e-2f);
            p = fmaf(y, p, 3.33333333e-1f);
            g = y * p;
        } else {
            g = aL + (x >= 0.0f ? h : hm) - 1.0f;
        }
    }
}

// FP32 spline table: per interval the cubic in the local coordinate
// t = (ln d - ln r_0) / h - k in [0, 1), coefficients pre-multiplied by
// log2(e) so that N = 2^(a + t (b + t (c + t d))): one 16-byte LDS read.
struct FastSpline {
    // The records run from rec[vmin], a constant one for ln d below ln r_0
    // (N = 2^-126, i.e. 0 to FP32 precision, S = 1), over the R - 1 intervals to
    // rec[vmax], constant above ln r_{R-1} (N = 1, S = 0); rec[0] starts at the
    // record boundary nearest to r.  v = log2(d / r) * inv_h2 + off is the
    // position: inv_h2 = ln 2 / h, off = the distance of r from that boundary
    // (0 on the evolution's grid, whose node r is).  Counted from r, a position
    // near r rounds to its own small size; counted from r_0 it would round by
    // up to 3e-5 of a record, which is 1e-6 of N.
    const float4* rec;
    float inv_h2, off, vmin, vmax;
};

// v clamped to the table by one median-of-three (log2_d is finite: it is the
// log of a distance); v - floor(v) is exact.
__device__ __forceinline__ float fspline_log2n(const FastSpline& s, float log2_d) {
    const float v = __builtin_amdgcn_fmed3f(fmaf(log2_d, s.inv_h2, s.off), s.vmin, s.vmax);
    const float t = __builtin_amdgcn_fractf(v);
    int k;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(k) : "v"(v));
    const float4 c = s.rec[k];
    return fmaf(t, fmaf(t, fmaf(t, c.w, c.z), c.y), c.x);
}

__device__ __forceinline__ float fspline_n(const FastSpline& s, float log2_d) {
    return fexp2(fspline_log2n(s, log2_d));
}

// S = 1 - N = -(2^p - 1) from p = log2 N near N = 1, where the subtraction
// would keep only the absolute precision of N: the series for |p ln 2| < 1/4
// (relative error < 2e-8).
constexpr float kNearOne = -0.360673760f;  // p above it: |p ln 2| < 1/4

__device__ __forceinline__ float fs_near_one(float p) {
    return -fexp2m1_small(p);
}

// Launch-invariant constants of the FP32 integrand, formed once per lane in
// vector registers: an FP32 operation with a scalar-register operand issues at
// half the rate of one with vector or literal operands.
struct Fp32Consts {
    float pi;
    float log2_r;
    float cut;         // 1e10 r^4
    float norm;        // Nc^2 / (8 pi^4), halved when symmetrised, times the caller's scale of the weights
    float mirror;      // 1 when symmetrised (the mirrored sample counts too), else 0
    float nf_over_nc;
    float mu;          // ln mu0 log2 e
    float right0;      // 5 (ln 4 C2 / Lambda^2) log2 e - 10 log2 r
    float b0;          // b0 0.2 ln 2
    bool wide;         // half-angle bins reach beyond 0.53 pi (the same for a whole block)
};

// The FP32 K2 + Kf integrand: the cancellation-free formula of
// nlo_integrand_stable with every distance in units of r, the transcendentals
// on the fast primitives above, logs of distances (base 2) from the log1p
// forms, N from the local-coordinate spline.  t1 = log2(z / r), t2 = log2(z' /
// r), y1 = theta / 2, y2 = theta' / 2 (modulo pi, in [-pi/2, pi/2] but for the
// bin across pi/2, which reaches up to pi).
//
// Issue-bound: the cost of a sample is its instructions, an FP32 add, mul or fma
// on vector registers or literals counting 2 cycles, min / max / compare /
// select / convert 4, a transcendental 8.  Hence the forms below: 4 sin^2 in
// one polynomial without a fold; the kernels from squared reciprocals (rcp
// for rsq and its squares); dipoles as n_z S_y' + (n_y' - n_y); and the rare
// cases (N near 1, the coupling near its freezing scale, the K2 cut, a
// non-finite value) behind tests that a whole wave takes or skips, which pays
// because the lanes of a wave hold neighbouring samples (sobol_order.hpp).
// 2^20 samples of 228 parents: 1.51 -> 1.17 ms (about 770 cycles a sample and
// wave; the listing counts 345 instructions before), and 2 to 5 times closer
// to the FP64 evaluation in most parents.
// SPLIT: the K2 and Kf parts are wanted apart.
template <bool ANYC, bool SPLIT>
__device__ __forceinline__ NloStable<float> nlo_integrand_fp32(const Fp32Consts& c, float t1, float t2, float y1,
                                                               float y2, const FastSpline& sp,
                                                               const NloCoupling<float>& cpl) {
    NloStable<float> out{0.0f, 0.0f, 0.0f};
    const float z = fexp2(t1), z2 = fexp2(t2);
    const float s1 = f4sin2(y1, c.pi), s2 = f4sin2(y2, c.pi), s3 = c.wide ? f4sin2_wide(y1 - y2, c.pi) : f4sin2(y1 - y2, c.pi);  // 4 sin^2
    const float zz2 = z * z2;
    float z1m = z - 1.0f, z2m = z2 - 1.0f;
    if (__any(fminf(fabsf(t1), fabsf(t2)) < 0.25f)) {  // 2^t - 1 near t = 0 without cancellation
        keep_branch(t1);
        z1m = fabsf(t1) < 0.25f ? fexp2m1_small(t1) : z1m;
        z2m = fabsf(t2) < 0.25f ? fexp2m1_small(t2) : z2m;
    }
    const float xsq = fmaf(z, s1, z1m * z1m);
    const float x2sq = fmaf(z2, s2, z2m * z2m);
    const float zsq = fmaf(zz2, s3, (z - z2) * (z - z2));
    if (!(fmin3(xsq, x2sq, zsq) >= 1e-37f)) return out;
    // log2(X / Y): (X^2 - z^2) / z^2 = rho (rho - 2 cos t), rho = r / z, cos t = 1 - 2 sin^2(t / 2)
    const float rho1 = frcp(z), rho2 = frcp(z2);
    const float u1 = rho1 * ((rho1 - 2.0f) + s1);
    const float u2 = rho2 * ((rho2 - 2.0f) + s2);
    const float lxy = fabsf(u1) < 0.5f ? fhalf_log2_1p_small(u1) : 0.5f * flog2(xsq) - t1;
    const float lx2y2 = fabsf(u2) < 0.5f ? fhalf_log2_1p_small(u2) : 0.5f * flog2(x2sq) - t2;
    const float log_x = t1 + lxy, log_x2 = t2 + lx2y2, log_zz = 0.5f * flog2(zsq);
    const float p_x = fspline_log2n(sp, log_x), p_y = fspline_log2n(sp, t1);
    const float p_x2 = fspline_log2n(sp, log_x2), p_y2 = fspline_log2n(sp, t2);
    const float n_x = fexp2(p_x), n_y = fexp2(p_y), n_x2 = fexp2(p_x2), n_y2 = fexp2(p_y2);
    const float n_z = fspline_n(sp, log_zz);
    float s_x = 1.0f - n_x, s_y = 1.0f - n_y, s_x2 = 1.0f - n_x2, s_y2 = 1.0f - n_y2;
    float dny = n_y2 - n_y, dnx = n_x - n_x2;
    float p_max = fmax2(fmax3(p_x, p_y, p_x2), p_y2);
    if (__any(p_max > kNearOne)) {
        keep_branch(p_max);
        s_x = p_x > kNearOne ? fs_near_one(p_x) : s_x;
        s_y = p_y > kNearOne ? fs_near_one(p_y) : s_y;
        s_x2 = p_x2 > kNearOne ? fs_near_one(p_x2) : s_x2;
        s_y2 = p_y2 > kNearOne ? fs_near_one(p_y2) : s_y2;
        // differences of amplitudes near 1 from the more accurate S
        if (fminf(p_y, p_y2) > kNearOne) dny = s_y - s_y2;
        if (fminf(p_x, p_x2) > kNearOne) dnx = s_x2 - s_x;
    }
    // S_X (S_Y - S_Z S_Y') and its mirror: S_Y - S_Z S_Y' = N_Z S_Y' + N_Y' - N_Y
    const float dip = s_x * fmaf(n_z, s_y2, dny);
    const float dips = s_x2 * fmaf(n_z, s_y, -dny);

    // L = ln(X Y' / (X' Y)) from its base-2 form
    const float L2 = lxy - lx2y2;
    const float x = (2.0f * kLn2f) * L2;  // 2 L
    float h, hm, g;
    fhg(x, 2.0f * L2, h, hm, g);
    const float ix = frcp(xsq), ix2 = frcp(x2sq), iz = frcp(zsq);
    const float zq = z * z, z2q = z2 * z2;
    const float B2 = z2q * iz * ix2, C2 = ix * ix2, D2 = zq * iz * ix;
    const float A = zz2 * iz;
    const float A2g = (2.0f * A) * (A * g);
    const float k = fmaf(x, D2, fmaf(h, fmaf(-4.0f, B2, C2), A2g));
    const float ks = fmaf(-x, B2, fmaf(hm, fmaf(-4.0f, D2, C2), A2g));
    float k2 = k * dip, k2s = ks * dips;
    // |K2| > 1e10 with |dipole| < 1e-10 (S/bk/derivatives.py:589), J = z^2 z'^2
    if (__any(fminf(fabsf(dip), fabsf(dips)) < 1e-10f)) {
        keep_branch(k2);
        const float cut = c.cut * (zq * z2q);
        if (fabsf(k) > cut && fabsf(dip) < 1e-10f) k2 = 0.0f;
        if (fabsf(ks) > cut && fabsf(dips) < 1e-10f) k2s = 0.0f;
    }
    const float kf = fmaf(h, B2, -A2g) * s_y, kfs = fmaf(hm, D2, -A2g) * s_y2;
    // smallest distance but r, whose logarithm is 0 here
    const float log_min = fmin3(fmin3(log_x, t1, log_x2), t2, log_zz);
    float as;
    if (!ANYC || cpl.mode == 0) {  // smooth coupling at the smallest distance (production)
        // in base 2: right = 5 (ln s0 - 2 ln d) log2 e, mu = ln mu0 log2 e,
        // alpha = 1 / (b0 0.2 ln 2 (max(mu, right) + log2(1 + 2^-|mu - right|)));
        // the last term is below half an ulp of the sum (>= 13) for |mu - right| > 22
        const float right = fmax2(fmaf(-10.0f, log_min, c.right0), c.right0);
        float den = fmax2(c.mu, right);
        float d = c.mu - right;
        if (__any(fabsf(d) < 22.0f)) {
            keep_branch(d);
            den += flog2(1.0f + fexp2(-fabsf(d)));
        }
        as = frcp(c.b0 * den);
    } else if (cpl.mode == 1) {
        as = cpl.as_const;
    } else {
        as = alpha_thresholds_log<float>((fminf(log_min, 0.0f) + c.log2_r) * kLn2f, cpl.log_4c2);
    }
    const float scale = (as * as) * c.norm;
    // Kf's dipole difference is df = n_x - n_x2 and its mirror
    float k2r = fmaf(c.mirror, k2s, k2), kfr = dnx * fmaf(-c.mirror, kfs, kf);
    out.total = fmaf(-c.nf_over_nc, kfr, k2r) * scale;
    const bool finite = isfinite(out.total);
    if (finite && !SPLIT) return out;
    if (c.mirror == 0.0f) {  // 0 times an infinite mirror image
        k2r = k2;
        kfr = dnx * kf;
    }
    k2r *= scale;
    kfr = c.nf_over_nc > 0.0f ? -c.nf_over_nc * kfr * scale : 0.0f;
    out.k2 = isfinite(k2r) ? k2r : 0.0f;
    out.kf = isfinite(kfr) ? kfr : 0.0f;
    if (!finite) out.total = out.k2 + out.kf;
    return out;
}

}  // namespace nlo
