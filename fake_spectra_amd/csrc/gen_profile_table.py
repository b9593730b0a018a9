"""Generate profile_table.h: G(u) = 1 - 2u D(u) (D: Dawson's integral) as cubics
in t = 16u^2 + 2, indexed by the bits of t.

G is the real-axis factor of the damping term of the Voigt function,
    Re w(u + ia) = exp(a^2 - u^2) cos(2au) - (2/sqrt(pi)) (a G(u) - a^3/6 D'''(u) + ...),
and an even entire function of u.  Every octave of t is cut into BINS equal
bins, so that a bin's number is the low exponent bits and the first mantissa
bits of t as a float, and its left edge is t with the other mantissa bits
cleared: neither core and wing nor small and large u need a case of their
own.  The 2 keeps t at or above an exponent whose low five bits are zero; the
16 makes it small against u^2 where the Gaussian, whose exponent is taken from
the same t, still matters (with 4u^2 + 2 the rounding of t cost the Gaussian
up to 1.6 times the error for u < 1).  Row r holds the four coefficients of the cubic in
t - edge (one 128-bit LDS read), a Chebyshev fit in float64 weighted by
1/|G|: within a bin t varies by at most 1/32 of itself, which holds the
truncation below 2e-8 of G (4.2e-8 of 0.01 next to its zero), less than the
float32 rounding that the evaluation adds (4.5e-8 rms).  A second table holds dG/d(u^2) the same way, for the
profile's derivative in the adjoint.  G comes from scipy.special.dawsn, beyond u = 9 from its
asymptotic series -sum_n (2n-1)!!/(2 u^2)^n.

Run:  python fake_spectra_amd/csrc/gen_profile_table.py > fake_spectra_amd/csrc/profile_table.h
"""
import numpy as np
from scipy.special import dawsn

OCTAVES = 32
BINS = 32
# The derivative's table holds 2^DSCALE dG/dp: its cubic coefficients fall as
# t^-5, below the float32 range without it.
DSCALE = 40


def g64(p):
    """G at u^2 = p."""
    u = np.sqrt(p)
    x = 1 / np.maximum(p, 1e-300)
    s = np.zeros_like(p)
    coef = np.cumprod([1.0] + [(2 * n - 1) / 2.0 for n in range(1, 16)])
    for n in range(15, 0, -1):
        s = (s + coef[n]) * x
    return np.where(u > 9.0, -s, 1 - 2 * u * dawsn(u))


def dg64(p):
    """dG/dp at u^2 = p: -(D/u + G), beyond u = 9 from the series."""
    u = np.sqrt(np.maximum(p, 1e-30))
    x = 1 / np.maximum(p, 1e-300)
    s = np.zeros_like(p)
    coef = np.cumprod([1.0] + [(2 * n - 1) / 2.0 for n in range(1, 16)])
    for n in range(15, 0, -1):
        s = (s + n * coef[n]) * x
    return np.where(u > 9.0, s * x, -dawsn(u) / u - (1 - 2 * u * dawsn(u)))


def rows(f, scale=1.0):
    th = np.cos(np.pi * (np.arange(24) + 0.5) / 24)
    out, worst = [], 0.0
    for e in range(1, OCTAVES + 1):
        w = 2.0 ** e / BINS
        for m in range(BINS):
            lo = 2.0 ** e + m * w
            floor = 0.01 if lo < 64 else 0.0
            g = f((lo + (th + 1) / 2 * w - 2) / 16)
            c = np.polynomial.chebyshev.chebfit(th, g, 3, w=1 / np.maximum(np.abs(g), floor))
            # a polynomial in t - lo
            mono = np.polynomial.Polynomial(np.polynomial.chebyshev.cheb2poly(c))(
                np.polynomial.Polynomial([-1.0, 2.0 / w])).coef
            v = np.linspace(0, w, 101)
            ref = f((lo + v - 2) / 16)
            err = np.abs(np.polyval(mono[::-1], v) - ref) / np.maximum(np.abs(ref), floor)
            worst = max(worst, float(err.max()))
            out.append(mono * scale)
    return out, worst


def main():
    r, worst = rows(g64)
    d, dworst = rows(dg64, 2.0 ** DSCALE)
    print("/* Generated by gen_profile_table.py; do not edit. */")
    print("/* G(u) = 1 - 2u D(u): cubics in t - edge, t = 16u^2 + 2, %d bins in each of %d octaves of t from 2" % (
        BINS, OCTAVES))
    print("   (max float64 fit error %.2g of G, of 0.01 near its zero), and 2^%d dG/d(u^2) (%.2g). */" % (worst, DSCALE, dworst))
    print("#pragma once")
    print("#define FSAMD_P_OCTAVES %d" % OCTAVES)
    print("#define FSAMD_P_BINS %d" % BINS)
    print("#define FSAMD_P_DSCALE %d" % DSCALE)
    for name, t in (("COEF", r), ("DCOEF", d)):
        print("/* initializer for a float[FSAMD_P_OCTAVES * FSAMD_P_BINS * 4] array */")
        print("#define FSAMD_P_%s_INIT { \\" % name)
        for c in t:
            print("    " + ", ".join("%.9ef" % v for v in c) + ", \\")
        print("}")


if __name__ == "__main__":
    main()
