"""Generate dawson64_table.h: float64 pieces of G(u) = 1 - 2u D(u) (D: Dawson's
integral) on [0, UMAX), for the FP64 Voigt profile at small damping
(voigt64_small, voigt.h).

Piece k holds the monomial coefficients in u - (k + 1/2) / PER_UNIT of a
Chebyshev fit of degree NCOEF - 1: the pieces are narrow (1/4), so the
truncation (about 1e-15) stays below the rounding of the evaluation.  D comes
from Rybicki's sum with step 0.2 in extended precision: sum over odd n of
exp(-(u - 0.2 n)^2) / n / sqrt(pi), accurate to exp(-(pi / 0.4)^2) ~ 1e-27.

Run:  python fake_spectra_amd/csrc/gen_dawson64_table.py > fake_spectra_amd/csrc/dawson64_table.h
"""
import numpy as np

PER_UNIT = 4
UMAX = 10
NCOEF = 12


def g(u):
    u = np.asarray(u, dtype=np.longdouble)
    n = np.arange(-401, 402, 2).astype(np.longdouble)
    h = np.longdouble(1) / 5
    d = (np.exp(-(u[..., None] - h * n) ** 2) / n).sum(-1) / np.sqrt(np.longdouble(np.pi))
    return 1 - 2 * u * d


def pieces():
    th = np.cos(np.pi * (np.arange(40) + 0.5) / 40)
    half = 0.5 / PER_UNIT
    out, worst = [], 0.0
    for k in range(UMAX * PER_UNIT):
        mid = (k + 0.5) / PER_UNIT
        c = np.polynomial.chebyshev.chebfit(th, g(mid + half * th).astype(np.float64), NCOEF - 1)
        mono = np.polynomial.chebyshev.cheb2poly(c) / half ** np.arange(NCOEF)
        v = np.linspace(-half, half, 81)
        ref = g(mid + v)
        val = np.polyval(mono[::-1].astype(np.longdouble), v.astype(np.longdouble))
        worst = max(worst, float(np.max(np.abs(val - ref))))
        out.append(mono)
    return out, worst


def main():
    rows, worst = pieces()
    print("/* Generated by gen_dawson64_table.py; do not edit. */")
    print("/* G(u) = 1 - 2u D(u) on [0, %d): %d pieces of width 1/%d (max error %.1g). */" % (
        UMAX, len(rows), PER_UNIT, worst))
    print("#pragma once")
    print("#define FSAMD_G64_PER_UNIT %d" % PER_UNIT)
    print("#define FSAMD_G64_UMAX %d.0" % UMAX)
    print("#define FSAMD_G64_NPIECE %d" % len(rows))
    print("#define FSAMD_G64_NCOEF %d" % NCOEF)
    print("/* initializer for a double[FSAMD_G64_NPIECE * FSAMD_G64_NCOEF] array */")
    print("#define FSAMD_G64_COEF_INIT { \\")
    for r in rows:
        print("    " + ", ".join("%.17e" % v for v in r) + ", \\")
    print("}")


if __name__ == "__main__":
    main()
