"""Generate exp_table.h: 2^(j/N) to twice float64 precision and the constants of
the argument reduction, for flux_exp (flux.hip).

With k = rint(x N / ln 2), r = x - k ln 2 / N: exp(x) = 2^(k / N) exp(r) and
2^(k/N) = 2^(k >> log2 N) T[k mod N] (the table-driven exponential of P. T. P.
Tang, ACM Trans. Math. Softw. 15, 1989).  ln 2 / N is split so that k times its
upper part is exact for |k| < 2^20.

Run:  python fake_spectra_amd/csrc/gen_exp_table.py > fake_spectra_amd/csrc/exp_table.h
"""
from decimal import Decimal, getcontext

N = 128
getcontext().prec = 60


def split(d):
    """d as the sum of two doubles, the first the nearest to d."""
    hi = float(d)
    return hi, float(d - Decimal(hi))


def main():
    ln2 = Decimal(2).ln()
    scale = 2 ** 39   # upper part: 33 bits of ln 2 / 128 = 2^-7.5
    up = float(int((ln2 / N) * scale * 2) / Decimal(scale * 2))
    print("/* Generated by gen_exp_table.py; do not edit. */")
    print("/* 2^(j/%d) as hi + lo, and the reduction by ln 2 / %d. */" % (N, N))
    print("#pragma once")
    print("#define FSAMD_EXP_N %d" % N)
    print("#define FSAMD_EXP_LOG2N %d" % (N.bit_length() - 1))
    print("#define FSAMD_EXP_INV %.17e" % float(N / ln2))
    print("#define FSAMD_EXP_STEP_HI %.17e" % up)
    print("#define FSAMD_EXP_STEP_LO %.17e" % float(ln2 / N - Decimal(up)))
    print("/* initializer for a double[2 * FSAMD_EXP_N] array */")
    print("#define FSAMD_EXP_INIT { \\")
    for j in range(N):
        hi, lo = split((ln2 * j / N).exp())
        print("    %.17e, %.17e%s \\" % (hi, lo, "," if j + 1 < N else ""))
    print("}")


if __name__ == "__main__":
    main()
