"""Calls at the ends of what the entry points take."""
import numpy as np
import pytest

from fake_spectra_amd import spectra_priv as SP
from gpu_util import dev
from test_gpu_edges import small_gas

pytestmark = pytest.mark.gpu

# sightlines in nearly all cells of the search grid, in some, in one
@pytest.mark.parametrize("nlos", [1, 30, 700])
def test_near_lines_of_supports_that_are_no_numbers(oracle, nlos):
    """Particles of infinite or undefined support are near no sightline, as in
    the neighbour lists, whatever the cell they lie in."""
    args = small_gas(900, 1000.0, nlos, 8, 1, 0.01)
    box, pos, h, axis, cofm = args[3], args[11], args[15], args[16], args[17]
    h[::5], h[1::5], h[2::5] = np.inf, np.nan, -np.inf
    pos[: min(nlos, 450)] = cofm[: min(nlos, 450)]      # in cells that hold a sightline
    finite = np.where(np.isfinite(h), h, np.float32(0))
    _, parts, _ = oracle.near_particles(box, pos, finite, axis, cofm)
    want = np.unique(parts[np.isfinite(h)[parts]])
    plan = SP.Plan(box, dev(pos), dev(h), dev(axis), dev(cofm))
    assert np.array_equal(plan.near_lines().cpu().numpy(), want)
    assert np.array_equal(SP._near_lines(box, pos, h, axis, cofm), want)
    plan.close()
