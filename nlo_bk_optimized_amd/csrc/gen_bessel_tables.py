"""Generate bessel_tables.inc (K0, K1 and the dilogarithm, for the DIS code)
and bessel_j1_i1_tables.inc (J1 and I1, for the K1 resummation).

For x > 2 the library evaluates K_nu(x) = e^(-x) / sqrt(x) * g_nu(s) with
s = 4 / x - 1 in (-1, 1], g_nu(s) = e^x sqrt(x) K_nu(x) (g_nu(-1) = sqrt(pi/2)).
g_nu is smooth on [-1, 1]; its Chebyshev interpolant at the N Chebyshev nodes
converges geometrically (degree 22: relative error 3e-17; degree 7: 1e-8).
The values come from mpmath's besselk at 40 digits.  FP64 evaluates the
degree-22 Chebyshev form; FP32 the degree-7 interpolant written in the power
basis of s for Horner's rule (float32 evaluation error 1.0e-7).  For
x <= 2 the four ascending series of K0 and K1 are tabulated as polynomials in
t = x^2 / 4 (exact rationals rounded once).

Dilogarithm: Li2(x) = u - u^2/4 + sum_k B_2k u^(2k+1) / (2k+1)!, u = -ln(1 - x),
for x in [-1, 1/2] (|u| <= ln 2); the coefficients B_2k / (2k+1)! are exact
rationals rounded once.

J1 (bessel_j1_i1_tables.inc): J1(x) / (x/2) on [0, 128) in 32 pieces of
width 4, each a degree-16 Chebyshev interpolant in s = (x - 4k)/2 - 1
(absolute error 1e-16).  I1 for x >= 8: e^-x sqrt(x) I1(x) as a degree-22
Chebyshev series in s = 16/x - 1 (relative error 5e-17).

Usage: python -m nlo_bk_optimized_amd.csrc.gen_bessel_tables (rewrites the .inc files)
"""

from __future__ import annotations

from pathlib import Path

import mpmath as mp

DEG64 = 22
DEG32 = 7
SERIES64, SERIES32 = 15, 8  # ascending-series terms for x <= 2 (t = x^2/4 <= 1)
J1_PIECES, J1_WIDTH, J1_DEG = 32, 4, 16
I1_DEG = 22
DILOG_TERMS = 10  # B_2 .. B_20: |term| < (ln 2 / 2 pi)^21 ~ 1e-20


def g(nu: int, s) -> mp.mpf:
    if s <= -1 + mp.mpf(10) ** -30:
        return mp.sqrt(mp.pi / 2)
    x = 4 / (s + 1)
    return mp.besselk(nu, x) * mp.exp(x) * mp.sqrt(x)


def chebyshev(nu: int, deg: int) -> list:
    n = deg + 1
    nodes = [mp.cos(mp.pi * (k + mp.mpf(1) / 2) / n) for k in range(n)]
    vals = [g(nu, s) for s in nodes]
    c = [2 * mp.fsum(vals[j] * mp.cos(mp.pi * m * (j + mp.mpf(1) / 2) / n) for j in range(n)) / n for m in range(n)]
    c[0] /= 2
    return c


def monomial(c: list) -> list:
    """Coefficients in the power basis of sum c_m T_m(s) (exact in mpmath)."""

    T = [[mp.mpf(1)], [mp.mpf(0), mp.mpf(1)]]
    for m in range(2, len(c)):
        a = [mp.mpf(0)] + [2 * v for v in T[m - 1]]
        b = T[m - 2] + [mp.mpf(0)] * (len(a) - len(T[m - 2]))
        T.append([x - y for x, y in zip(a, b)])
    mono = [mp.mpf(0)] * len(c)
    for m, cm in enumerate(c):
        for k, v in enumerate(T[m]):
            mono[k] += cm * v
    return mono


def chebyshev_interval(f, a, b, deg: int) -> list:
    n = deg + 1
    nodes = [mp.cos(mp.pi * (k + mp.mpf(1) / 2) / n) for k in range(n)]
    vals = [f((b - a) / 2 * t + (a + b) / 2) for t in nodes]
    c = [2 * mp.fsum(vals[j] * mp.cos(mp.pi * m * (j + mp.mpf(1) / 2) / n) for j in range(n)) / n for m in range(n)]
    c[0] /= 2
    return c


def j1_i1_tables() -> str:
    def j1h(x):
        return mp.besselj(1, x) / (x / 2) if x != 0 else mp.mpf(1)

    def i1s(t):
        if t <= -1 + mp.mpf(10) ** -30:
            return 1 / mp.sqrt(2 * mp.pi)
        x = 16 / (t + 1)
        return mp.besseli(1, x) * mp.exp(-x) * mp.sqrt(x)

    lines = ["// Generated by gen_bessel_tables.py: J1(x)/(x/2) on [0, 128) in 32 pieces of width 4",
             "// (degree-16 Chebyshev in s = (x - 4k)/2 - 1) and e^-x sqrt(x) I1(x) for x >= 8",
             "// (degree-22 Chebyshev in s = 16/x - 1)."]
    lines.append(f"constexpr int kJ1Pieces = {J1_PIECES}, kJ1Deg = {J1_DEG};")
    rows = []
    for k in range(J1_PIECES):
        c = chebyshev_interval(j1h, mp.mpf(J1_WIDTH * k), mp.mpf(J1_WIDTH * (k + 1)), J1_DEG)
        rows.append(", ".join(mp.nstr(v, 21, min_fixed=-1, max_fixed=-1) for v in c))
    lines.append(f"__device__ constexpr double kJ1Cheb[{J1_PIECES * (J1_DEG + 1)}] = {{\n    " + ",\n    ".join(rows) + "};")
    c = chebyshev_interval(i1s, mp.mpf(-1), mp.mpf(1), I1_DEG)
    lines.append(f"constexpr int kI1Deg = {I1_DEG};")
    lines.append(f"__device__ constexpr double kI1Cheb[{I1_DEG + 1}] = {{\n    " +
                 ",\n    ".join(mp.nstr(v, 21, min_fixed=-1, max_fixed=-1) for v in c) + "};")
    return "\n".join(lines) + "\n"


def main() -> None:
    mp.mp.dps = 40
    lines = [
        "// Generated by gen_bessel_tables.py: g_nu(s) = e^x sqrt(x) K_nu(x), s = 4/x - 1,",
        "// for x > 2 (FP64: Chebyshev coefficients, sum c_m T_m(s); FP32: power basis).",
    ]
    for nu in (0, 1):
        c = chebyshev(nu, DEG64)
        body = ",\n    ".join(mp.nstr(v, 21, min_fixed=-1, max_fixed=-1) for v in c)
        lines.append(f"constexpr int kBesselK{nu}Deg64 = {DEG64};")
        lines.append(f"__device__ constexpr double kBesselK{nu}Cheb64[{DEG64 + 1}] = {{\n    {body}}};")
    # FP32, x > 2: the degree-7 interpolant in the monomial basis of s
    # (Horner: one fma per degree; float32 evaluation error 1.0e-7)
    for nu in (0, 1):
        mono = monomial(chebyshev(nu, DEG32))
        body = ",\n    ".join(mp.nstr(v, 10, min_fixed=-1, max_fixed=-1) + "f" for v in mono)
        lines.append(f"constexpr int kBesselK{nu}Deg32 = {DEG32};")
        lines.append(f"__device__ constexpr float kBesselK{nu}Mono32[{DEG32 + 1}] = {{\n    {body}}};")
    from fractions import Fraction
    from math import comb, factorial

    # x <= 2: the ascending series as polynomials in t = x^2/4 (Horner), the
    # exact rational coefficients rounded once:
    #   I0 = sum t^k/k!^2, S0 = sum H_k t^k/k!^2,
    #   I1 = sum t^k/(k!(k+1)!), S1 = sum (H_k + H_(k+1)) t^k/(k!(k+1)!)
    def harmonic(k):
        return sum((Fraction(1, j) for j in range(1, k + 1)), Fraction(0))

    for terms, typ, name, suffix in ((SERIES64, "double", "64", ""), (SERIES32, "float", "32", "f")):
        rows = {
            "I0": [Fraction(1, factorial(k) ** 2) for k in range(terms)],
            "S0": [harmonic(k) / factorial(k) ** 2 for k in range(terms)],
            "I1": [Fraction(1, factorial(k) * factorial(k + 1)) for k in range(terms)],
            "S1": [(harmonic(k) + harmonic(k + 1)) / (factorial(k) * factorial(k + 1)) for k in range(terms)],
        }
        lines.append(f"constexpr int kBesselSeriesTerms{name} = {terms};")
        for key, coef in rows.items():
            body = ",\n    ".join(
                (repr(float(c)) if typ == "double" else mp.nstr(mp.mpf(c.numerator) / c.denominator, 10, min_fixed=-1, max_fixed=-1) + suffix)
                for c in coef)
            lines.append(f"__device__ constexpr {typ} kBesselSeries{key}_{name}[{terms}] = {{\n    {body}}};")

    B = [Fraction(1)]
    for m in range(1, 2 * DILOG_TERMS + 1):
        B.append(-sum(comb(m + 1, k) * B[k] for k in range(m)) / Fraction(m + 1))
    coef = [B[2 * k] / factorial(2 * k + 1) for k in range(1, DILOG_TERMS + 1)]
    body = ",\n    ".join(repr(float(c)) for c in coef)
    lines.append(f"constexpr int kDilogTerms = {DILOG_TERMS};")
    lines.append(f"__device__ constexpr double kDilogBernoulli[{DILOG_TERMS}] = {{\n    {body}}};")
    out = Path(__file__).with_name("bessel_tables.inc")
    out.write_text("\n".join(lines) + "\n")
    print(f"wrote {out}")
    out2 = Path(__file__).with_name("bessel_j1_i1_tables.inc")
    out2.write_text(j1_i1_tables())
    print(f"wrote {out2}")


if __name__ == "__main__":
    main()
