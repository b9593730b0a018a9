"""Generate dawson_table.h: piecewise polynomials for G(u) = 1 - 2u D(u).

No kernel reads this table since profile_table.h took its place; the tests
of the generated tables still check it against Dawson's integral.

D is Dawson's integral; G(u) is D'(u), the real-axis factor of the first
term of the Voigt function's expansion in the damping parameter a:
    Re w(u + ia) = exp(a^2 - u^2) cos(2au) - (2/sqrt(pi)) (a G(u) - a^3/6 D'''(u) + ...)

Rows of FSAMD_G_STRIDE floats (16-byte aligned, so that a row loads with two
128-bit reads; 12 floats rather than 8, so that rows that share LDS banks
are 8 apart instead of 4: fewer bank conflicts between the lanes of a
wavefront reading different rows, measured 0.7-1.9% faster deposits):
  rows 0..NPIECE-1 (u in [0, UMAX)): piece k holds the monomial coefficients
    of G in s = (u - k WIDTH) / WIDTH in [0, 1) (the fractional part of
    u / WIDTH), degree DEG, from a Chebyshev interpolant in float64 against
    scipy.special.dawsn on the piece;
  row NPIECE (u >= UMAX): G itself as a polynomial of degree DEG in
    x = 1/u^2 with no constant term, G = x R(x), R of degree DEG - 1 with
    R(0) = -1/2 (the asymptotic series G ~ -sum_k (2k-1)!!/2^k x^k) and the
    other coefficients fitted by least squares in relative error over
    x in (0, 1/UMAX^2] (as accurate as a degree-DEG R: both fits sit at the
    2e-8 noise of the float64 reference).  Every row is then evaluated the
    same way, by Horner in its variable (s or x), with no final product.

Run:  python fake_spectra_amd/csrc/gen_dawson_table.py > fake_spectra_amd/csrc/dawson_table.h
"""
import numpy as np
from scipy.special import dawsn

WIDTH = 0.25
DEG = 6
UMAX = 7.0
STRIDE = 12


def g64(u):
    return 1 - 2 * u * dawsn(u)


def core_rows():
    npiece = int(round(UMAX / WIDTH))
    tn = np.cos(np.pi * (np.arange(64) + 0.5) / 64)
    rows, worst = [], 0.0
    for p in range(npiece):
        lo = p * WIDTH
        u = lo + (tn + 1) / 2 * WIDTH
        c = np.polynomial.chebyshev.chebfit(tn, g64(u), DEG)
        # monomials in t = 2s - 1, then composed with t(s)
        mono = np.polynomial.Polynomial(np.polynomial.chebyshev.cheb2poly(c))(
            np.polynomial.Polynomial([-1.0, 2.0])).coef
        ss = np.linspace(0, 1, 1001)
        uu = lo + ss * WIDTH
        worst = max(worst, np.max(np.abs(np.polyval(mono[::-1], ss) - g64(uu))))
        rows.append(mono)
    return rows, worst


def wing_row():
    x = np.linspace(1e-8, 1 / UMAX ** 2, 4000)
    r = g64(1 / np.sqrt(x)) / x
    a = np.stack([x ** k for k in range(1, DEG)], 1)
    c, *_ = np.linalg.lstsq(a / r[:, None], (r + 0.5) / r, rcond=None)
    rr = np.concatenate([[-0.5], c])          # R(x), degree DEG - 1
    fit = np.polynomial.polynomial.polyval(x, rr)
    return np.concatenate([[0.0], rr]), np.max(np.abs(fit - r) / np.abs(r))   # G(x) = x R(x)


def main():
    rows, worst = core_rows()
    wing, wworst = wing_row()
    npiece = len(rows)
    print("/* Generated by gen_dawson_table.py; do not edit. */")
    print("/* G(u) = 1 - 2u D(u): %d pieces of width %.3f, degree %d, on [0, %.2f) (max float64 fit" % (
        npiece, WIDTH, DEG, UMAX))
    print("   error %.3g), then G = x R(x), x = 1/u^2, for u >= %.2f, stored as a polynomial in x (max relative fit error %.3g). */" % (
        worst, UMAX, wworst))
    print("#pragma once")
    print("#define FSAMD_G_NPIECE %d" % npiece)
    print("#define FSAMD_G_DEG %d" % DEG)
    print("#define FSAMD_G_STRIDE %d" % STRIDE)
    print("#define FSAMD_G_NROW %d" % (npiece + 1))
    print("#define FSAMD_G_WIDTH %sf" % repr(float(WIDTH)))
    print("#define FSAMD_G_UMAX %sf" % repr(float(UMAX)))
    print("/* initializer for a float[FSAMD_G_NROW * FSAMD_G_STRIDE] array */")
    print("#define FSAMD_G_COEF_INIT { \\")
    pad = ", 0.0f" * (STRIDE - DEG - 1)
    for p, r in enumerate(rows):
        print("    " + ", ".join("%.9ef" % v for v in r) + pad + ",  /* u in [%.2f, %.2f) */ \\" % (
            p * WIDTH, (p + 1) * WIDTH))
    print("    " + ", ".join("%.9ef" % v for v in wing) + pad + ",  /* u >= %.2f: G(x) = x R(x) */ \\" % UMAX)
    print("}")


if __name__ == "__main__":
    main()
