"""profile_table.h (the FP32 profile's cubics of G = 1 - 2u D in t = 16u^2 + 2)
on the CPU: the header is its generator's output, and rows addressed by the
bits of t as voigt_terms does follow scipy's dawsn."""
import os
import re
import subprocess
import sys

import numpy as np
import pytest
from scipy.special import dawsn

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fake_spectra_amd", "csrc")


@pytest.fixture(scope="module")
def table():
    text = open(os.path.join(CSRC, "profile_table.h")).read()
    out = subprocess.run([sys.executable, os.path.join(CSRC, "gen_profile_table.py")], capture_output=True, text=True,
                         check=True)
    assert out.stdout == text
    octaves, bins = (int(re.search(r"#define FSAMD_P_%s (\d+)" % k, text).group(1)) for k in ("OCTAVES", "BINS"))
    c = np.array([float(v.strip().rstrip("f")) for v in
                  re.search(r"INIT \{(.*?)\n\}", text, re.S).group(1).replace("\\", "").split(",") if v.strip()])
    assert bins == 32 and c.size == octaves * bins * 4
    return c.astype(np.float32).reshape(-1, 4), octaves


# next to 0, around G's zero, core, transition, wing, and the last octaves
@pytest.mark.parametrize("lo,hi", [(0.0, 0.8), (0.8, 1.1), (1.1, 4.0), (4.0, 8.0), (8.0, 20.0), (20.0, 300.0),
                                   (300.0, 2.3e4)])
def test_rows_follow_dawson(table, lo, hi):
    coef, octaves = table
    u = np.linspace(lo, hi, 40001)
    t = (16.0 * u * u + 2.0).astype(np.float32)
    edge = t.view(np.uint32) & np.uint32(0xFFFC0000)
    row = ((edge >> 14) & np.uint32(0x3FFF)) // 16
    assert row.max() < octaves * 32
    d = t.astype(np.float64) - edge.view(np.float32)
    c = coef[row].astype(np.float64)
    got = c[:, 0] + d * (c[:, 1] + d * (c[:, 2] + d * c[:, 3]))
    uu = np.sqrt(np.maximum((t.astype(np.float64) - 2.0) / 16.0, 0.0))
    x = 1.0 / np.maximum(uu * uu, 1e-300)
    series = -0.5 * x * (1 + 1.5 * x * (1 + 2.5 * x * (1 + 3.5 * x * (1 + 4.5 * x * (1 + 5.5 * x * (1 + 6.5 * x))))))
    ref = np.where(uu < 12.0, 1.0 - 2.0 * uu * dawsn(uu), series)
    # the fit's 2e-8 (4.2e-8 of 0.01 around the zero), the FP32 rounding of four
    # coefficients whose terms are at most 1, 1/32, .. of G (6e-8), and half of
    # that again where the first terms are larger than G
    assert np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 0.05 if hi < 1.2 else 0.0)) < 1.2e-7
