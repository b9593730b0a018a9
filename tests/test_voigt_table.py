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
    c = [np.array([float(v.strip().rstrip("f")) for v in m.replace("\\", "").split(",") if v.strip()])
         for m in re.findall(r"COEF_INIT \{(.*?)\n\}", text, re.S)]
    assert bins == 32 and len(c) == 2 and all(x.size == octaves * bins * 4 for x in c)
    # as float64: a host library may flush FP32 denormals, which the last octave's
    # cubic terms are (the GPU keeps them)
    return [x.reshape(-1, 4) for x in c], octaves


# next to 0, around G's zero, core, transition, wing, and the last octaves
@pytest.mark.parametrize("lo,hi", [(0.0, 0.8), (0.8, 1.1), (1.1, 4.0), (4.0, 8.0), (8.0, 20.0), (20.0, 300.0),
                                   (300.0, 2.3e4)])
def test_rows_follow_dawson(table, lo, hi):
    (coef, dcoef), octaves = table
    u = np.linspace(lo, hi, 40001)
    t = (16.0 * u * u + 2.0).astype(np.float32)
    edge = t.view(np.uint32) & np.uint32(0xFFFC0000)
    row = ((edge >> 14) & np.uint32(0x3FFF)) // 16
    assert row.max() < octaves * 32
    d = t.astype(np.float64) - edge.view(np.float32)
    c = coef[row]
    got = c[:, 0] + d * (c[:, 1] + d * (c[:, 2] + d * c[:, 3]))
    uu = np.sqrt(np.maximum((t.astype(np.float64) - 2.0) / 16.0, 0.0))
    x = 1.0 / np.maximum(uu * uu, 1e-300)
    series = -0.5 * x * (1 + 1.5 * x * (1 + 2.5 * x * (1 + 3.5 * x * (1 + 4.5 * x * (1 + 5.5 * x * (1 + 6.5 * x))))))
    ref = np.where(uu < 12.0, 1.0 - 2.0 * uu * dawsn(uu), series)
    # the fit's 2e-8 (4.2e-8 of 0.01 around the zero), the FP32 rounding of four
    # coefficients whose terms are at most 1, 1/32, .. of G (6e-8), and half of
    # that again where the first terms are larger than G
    assert np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 0.05 if hi < 1.2 else 0.0)) < 1.2e-7
    # dG/d(u^2) = -(D/u + G), which cancels to 1/(2 u^4) at large u; zero at u = 1.502
    c = dcoef[row] * 2.0 ** -40
    got = c[:, 0] + d * (c[:, 1] + d * (c[:, 2] + d * c[:, 3]))
    series = 0.5 * x * x * (1 + 3 * x * (1 + 15 / 4 * x * (1 + 14 / 3 * x * (1 + 45 / 8 * x * (1 + 33 / 5 * x)))))
    us = np.maximum(uu, 1e-9)
    ref = np.where(uu < 12.0, -dawsn(us) / us - (1.0 - 2.0 * us * dawsn(us)), series)
    # 4e-8 of the fit (its terms fall as 1, 2/32, 3/32^2), the rounding as above
    assert np.max(np.abs(got - ref) / np.maximum(np.abs(ref), 0.05 if hi < 8.0 else 0.0)) < 2.0e-7
