"""exp_table.h (flux_exp's table and reduction, flux.hip) on the CPU: the header
is its generator's output, and its arithmetic restated here follows exp to
half an ulp and the two roundings before the last, 2^-7 of one each at most."""
import os
import re
import subprocess
import sys

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fake_spectra_amd", "csrc")


def test_header_is_generator_output_and_follows_exp():
    text = open(os.path.join(CSRC, "exp_table.h")).read()
    out = subprocess.run([sys.executable, os.path.join(CSRC, "gen_exp_table.py")], capture_output=True, text=True,
                         check=True)
    assert out.stdout == text
    inv, hi, lo = (float(re.search(r"#define FSAMD_EXP_%s (\S+)" % k, text).group(1)) for k in ("INV", "STEP_HI", "STEP_LO"))
    tab = np.array([float(v) for v in re.search(r"INIT \{(.*?)\n\}", text, re.S).group(1).replace("\\", "").split(",")
                    if v.strip()]).reshape(-1, 2)
    wide = np.longdouble

    def fma(a, b, c):    # 64 bits of mantissa hold the product but for its last bits
        return (wide(a) * wide(b) + wide(c)).astype(np.float64)

    x = -np.concatenate([np.linspace(0, 700, 200001), np.geomspace(1e-17, 1, 1000)])
    kf = np.rint(x * inv)
    r = fma(kf, -lo, fma(kf, -hi, x))
    q = fma(r, 1 / 120, 1 / 24)
    q = fma(r, q, 1 / 6)
    q = fma(r, q, 0.5)
    q = fma(r * r, q, r)
    T = tab[kf.astype(int) % 128]
    got = np.ldexp(T[:, 0] + fma(T[:, 0], q, T[:, 1]), kf.astype(int) // 128)
    ref = np.exp(wide(x))
    ulp = np.spacing(ref.astype(np.float64)).astype(wide)
    assert np.max(np.abs(got - ref) / ulp) < 0.5 + 2 * 2.0 ** -7
