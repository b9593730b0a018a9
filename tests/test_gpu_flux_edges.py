"""Flux statistics at the sizes where the kernels' splits change: the mean-flux
iteration on fields with excluded, negative and deep pixels."""
import math

import numpy as np
import pytest
import torch

import fluxstats as FS
from fake_spectra_amd import fluxstatistics as GF

pytestmark = pytest.mark.gpu


def _field(nlos, npix, seed):
    r = np.random.default_rng(seed)
    t = np.exp(1.5 * r.standard_normal((nlos, npix)) - 1)
    t[r.random(t.shape) < 0.05] = 0.0
    t[r.random(t.shape) < 0.01] = 1e5     # no flux left
    return t


@pytest.mark.parametrize("n", [1, 2, 255, 257, 1536 * 256 - 1, 1536 * 256 * 2, 1536 * 256 * 5 + 77])
@pytest.mark.parametrize("target", [0.35, 0.68, 0.9])
@pytest.mark.parametrize("tol", [1e-2, 1e-5, 1e-10])
def test_mean_flux_steps_as_newton(n, target, tol):
    """The iterates are Newton's from 1 whichever moments served a step (1e-14
    each): the same number of steps, so the same scale even for a coarse tol.
    Sums of 2e6 terms: 1e-13; the bound has 10 for the steps."""
    t = _field(1, n, n)[0] if n > 2 else np.array([0.3, 2.0])[:n]
    got, ref = GF.mean_flux(torch.from_numpy(t).cuda(), target, tol), FS.mean_flux_scale(t, target, tol)
    assert abs(got - ref) <= 1e-12 * ref


def test_mean_flux_excluded_and_negative_pixels():
    r = np.random.default_rng(5)
    t = np.exp(r.standard_normal(400000))
    t[::7] = 50.0
    t[3::1000] *= -0.01
    for thresh in (10.0, 1e30):
        got = GF.mean_flux(torch.from_numpy(t).cuda(), 0.5, 1e-8, thresh)
        assert abs(got - FS.mean_flux_scale(t, 0.5, 1e-8, thresh=thresh)) <= 1e-12 * got
    t[11] = np.nan
    assert math.isnan(GF.mean_flux(torch.from_numpy(t).cuda(), 0.5))
