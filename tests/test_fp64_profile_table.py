"""dawson64_table.h (the FP64 profile's pieces of G = 1 - 2u D(u)) on the CPU:
the header is its generator's output, and the pieces follow scipy's dawsn to
the rounding of 1 - 2u D (eps times 2u D <= 1.1, and eps again)."""
import os
import re
import subprocess
import sys

import numpy as np
from scipy.special import dawsn

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fake_spectra_amd", "csrc")


def test_header_is_generator_output_and_follows_dawson():
    text = open(os.path.join(CSRC, "dawson64_table.h")).read()
    out = subprocess.run([sys.executable, os.path.join(CSRC, "gen_dawson64_table.py")], capture_output=True, text=True,
                         check=True)
    assert out.stdout == text
    per, ncoef = (int(re.search(r"#define FSAMD_G64_%s (\d+)" % k, text).group(1)) for k in ("PER_UNIT", "NCOEF"))
    c = np.array([float(v) for v in re.search(r"INIT \{(.*?)\n\}", text, re.S).group(1).replace("\\", "").split(",")
                  if v.strip()]).reshape(-1, ncoef)
    for k, row in enumerate(c):
        v = np.linspace(-0.5, 0.5, 65)[:-1] / per
        u = (k + 0.5) / per + v
        r = np.zeros_like(v)
        for x in row[::-1]:
            r = r * v + x
        assert np.max(np.abs(r - (1 - 2 * u * dawsn(u)))) < 1.5e-15
