"""Calls at the ends of what the entry points take."""
import numpy as np
import pytest
import torch

from fake_spectra_amd import _native as N, spectra_priv as SP, synth
from fake_spectra_amd.lines import HI_1215
from gpu_util import assert_tau_close, dev
from test_gpu_edges import small_gas
from torch_reference import BOLTZMANN, LIGHT, PROTONMASS, SIGMA_T, kernel_weight

pytestmark = pytest.mark.gpu

VELFAC = synth.Cosmology().velfac()


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


class LoneParticle:
    """One particle on one sightline in a box of twelve of its supports, a
    support of `support` Doppler widths (b = 10 km/s) and a damping parameter
    a; the density is so high that no pixel of the row ends a window."""

    def __init__(self, support, kernel, a):
        px = min(20.0, support / 50.0)                       # pixel in Doppler widths
        self.nbins, self.kernel = 2 * int(6 * support / px), kernel
        b0 = 10.0
        box = 12.0 * support * b0 / VELFAC
        pos = np.full((1, 3), 0.5 * box, dtype=np.float32)
        self.h = np.array([support * b0 / VELFAC], dtype=np.float32)
        cofm = np.array([[0.0, 0.5 * box + 0.2 * support * b0 / VELFAC, 0.5 * box]])
        temp = np.array([1e4 * (b0 / 12.85) ** 2], dtype=np.float32)
        gamma = a * b0 * 4 * np.pi * 1e5 / HI_1215.lambda_cm
        self.line = (HI_1215.lambda_cm, gamma, HI_1215.fosc, HI_1215.amumass)
        self.box, self.pos, self.cofm, self.temp = box, pos, cofm, temp
        self.dens = np.array([1e30], dtype=np.float32)
        self.plan = SP.Plan(box, dev(pos), dev(self.h), dev(np.array([1], dtype=np.int32)), dev(cofm))
        self.args = (self.nbins, kernel, VELFAC, dev(np.zeros((1, 3), dtype=np.float32)), dev(temp), [self.line],
                     [dev(self.dens)])
        # pixel centres from the particle, in supports
        self.at = ((np.arange(self.nbins) + 0.5) * box / self.nbins - float(pos[0, 0])) / float(self.h[0])

    def far_gradients(self, weights):
        """dL/d dens, dL/dT and dL/d vel of L = sum(weights tau) over pixels of the far
        wing, in FP64: with w(z) = i/sqrt(pi) sum_n c_n z^(-2n-1), z = u + ia, the sums
        of H = Re w, dH/du = Re w' and H + u dH/du + a dH/da = Re(w + z w') term by term
        (the last has lost 1/u^2 of its parts, which no difference of them keeps)."""
        lam, gamma, fosc, amu = self.line
        T, dens, h = float(self.temp[0]), float(self.dens[0]), float(self.h[0])
        b = np.sqrt(2 * BOLTZMANN / (amu * PROTONMASS)) / 1e5 * np.sqrt(T)
        a = gamma * lam / (4 * np.pi) / 1e5 / b
        amp = np.sqrt(3 * np.pi * SIGMA_T / 8) * lam * fosc / np.sqrt(np.pi) * (LIGHT / 1e5 / b)
        d2 = (float(self.pos[0, 1]) - self.cofm[0, 1]) ** 2 + (float(self.pos[0, 2]) - self.cofm[0, 2]) ** 2
        vh = VELFAC * np.sqrt(h * h - d2)
        dvk = vh / 4
        vv = np.arange(1, 8) * dvk - vh
        W = kernel_weight(self.kernel, np.sqrt(VELFAC ** 2 * d2 + vv * vv) / (VELFAC * h))
        width = self.box * VELFAC / self.nbins
        npts = 1 if width < b / 2 else int(2 * np.ceil(width / b) + 1)
        off = np.array([0.5]) if npts == 1 else np.arange(npts) / (npts - 1)
        t = np.ones(npts)
        if npts > 1:
            t[[0, -1]] = 0.5
            t /= npts - 1
        S = np.zeros(3)
        for z in np.nonzero(weights)[0]:
            v = (z + off) * width - VELFAC * float(self.pos[0, 0])
            zz = (vv[:, None] - v[None, :]) / b + 1j * a
            term, c, s = 1 / zz, 1.0, np.zeros((3,) + zz.shape, dtype=complex)
            for n in range(12):
                s[0] += c * term
                s[1] += -2 * n * c * term
                s[2] += -(2 * n + 1) * c * term / zz
                term, c = term / (zz * zz), c * (n + 0.5)
            S += weights[z] * np.einsum("i,j,kij->k", W, t, (1j / np.sqrt(np.pi) * s).real)
        scale = amp * dvk / VELFAC
        return S[0] * scale, -S[1] * scale * dens / (2 * T), S[2] * scale * dens / b

    def check(self):
        """tau everywhere (FP64 path) and the gradients of a side of the far wing
        alone, to the stated tolerance of tau."""
        self.plan.keep_windows(True)
        tau = SP.tau(self.plan, *self.args)[0].cpu().numpy()
        # the expansion begins near 2.25; the row's last pixel may be the other walk's, one box length off
        w = np.where((self.at > 2.4) & (self.at < 5.9), 1.0 + 0.3 * np.sin(7.0 * self.at), 0.0)
        got = SP.tau_adjoint(self.plan, *self.args, [dev(w[None])])
        SP.set_fp64(True)
        try:
            want = SP.tau(self.plan, *self.args)[0].cpu().numpy()
        finally:
            SP.set_fp64(False)
        assert np.all(want > 0) and np.max(np.abs(tau - want) / want) <= 1e-5
        for name, x, y in zip(("dens", "T", "vel"), (got[0][0][0], got[1][0], got[2][0, 0]), self.far_gradients(w)):
            assert abs(float(x) - y) <= 1e-5 * abs(y), name
        self.plan.close()


# supports at which powers of the far wing's distance leave the range of FP32
# numbers one after the other; weights flat and falling
@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("support", [10, 30, 100, 300, 1000, 3000])
def test_far_wing_of_wide_supports(support, kernel):
    LoneParticle(support, kernel, 1e-2).check()


# damping parameters up to where the optical depth drops the a^3 term, and beyond;
# supports of half a Doppler width and of twenty
@pytest.mark.parametrize("support,peak", [(0.5, 1e4), (3.0, 1e6), (20.0, 1e6)])
@pytest.mark.parametrize("a", [4e-4, 1.2e-3, 1.95e-3, 2.5e-3])
def test_saturated_gradients_keep_the_cubic_term(a, support, peak):
    """Gradients of sum(exp(-2 tau)) through saturated cores come from |u| = 3 to 5
    alone, where the a^3 term is up to 5.5e-7 of the profile, or from the wings: FP32
    against FP64, half of the density's are right to an FP32 unit in the last
    place, 2^-23, and half of the temperature's, a difference, to the stated 1e-5."""
    errs = [], []
    b0, n, nlos = 10.0, 300, 60
    for seed in range(4):
        rng = np.random.default_rng(seed)
        b = np.maximum(b0 * np.exp(0.02 * rng.standard_normal(n)), 0.9 * b0)
        temp = (1e4 * (b / 12.85) ** 2).astype(np.float32)
        h0 = support * b0 / VELFAC
        box = max(20 * h0, 40 * b0 / VELFAC)
        nbins = int(box * VELFAC / 2.5)
        pos = (rng.random((n, 3)) * box).astype(np.float32)
        h = (h0 * np.exp(0.2 * rng.standard_normal(n))).astype(np.float32)
        vel = (10 * rng.standard_normal((n, 3))).astype(np.float32)
        axis = (1 + np.arange(nlos) % 3).astype(np.int32)
        cofm = pos[rng.integers(0, n, nlos)].astype(np.float64) + 0.1 * h0
        line = (HI_1215.lambda_cm, a * b0 * 4 * np.pi * 1e5 / HI_1215.lambda_cm, HI_1215.fosc, HI_1215.amumass)
        plan = SP.Plan(box, dev(pos), dev(h), dev(axis), dev(cofm))
        plan.keep_windows(True)
        dens = np.exp(20 + 0.3 * rng.standard_normal(n)).astype(np.float32)
        call = (nbins, 1, VELFAC, dev(vel), dev(temp), [line])
        top = float(SP.tau(plan, *call, [dev(dens)])[0].max())
        dens = dev((dens * (peak / top)).astype(np.float32))
        grads, weights = [], None
        for fp64 in (True, False):
            SP.set_fp64(fp64)
            try:
                tau = SP.tau(plan, *call, [dens])[0]
                weights = -2 * torch.exp(-2 * tau) if weights is None else weights
                gd, gt, _ = SP.tau_adjoint(plan, *call, [dens], [weights])
            finally:
                SP.set_fp64(False)
            grads.append((gd[0].cpu().numpy(), gt.cpu().numpy()))
        for e, want, got in zip(errs, *grads):
            m = want != 0
            e.append(np.abs(got - want)[m] / np.abs(want[m]))
        plan.close()
    density, temperature = (np.concatenate(e) for e in errs)
    assert density.size > 200
    assert np.median(density) <= 2.0 ** -23 and np.median(temperature) <= 1e-5


def fp64_pairs(call):
    """A tau call's result and the pairs it walked in FP64."""
    N.check(N.lib().fsamd_set_stats(1))
    try:
        out = call()
        st = SP.last_stats()
    finally:
        N.check(N.lib().fsamd_set_stats(0))
    assert st["pairs"] > 0
    return out, st["fp64_pairs"]


# supports whose samples leave the profile's table (near 7600 Doppler widths), by
# little and by much
@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("support", [7600, 8000, 30000])
def test_far_wing_beyond_the_profile_table(support, kernel):
    lone = LoneParticle(support, kernel, 1e-2)
    assert fp64_pairs(lambda: SP.tau(lone.plan, *lone.args))[1] == 0
    lone.check()


# and beside narrow supports of the same rows; light and full profiles
@pytest.mark.parametrize("group", [16, 64])
@pytest.mark.parametrize("kernel", [0, 1, 3])
@pytest.mark.parametrize("a", [1e-4, 1e-2])
def test_supports_beyond_the_profile_table(oracle, a, kernel, group):
    n, nlos, nbins = 120, 6, 3000
    args = list(small_gas(n, 60000.0 / VELFAC, nlos, nbins, kernel, 0.02))
    args[14][:] = 1e4 * (30.0 / 12.85) ** 2
    args[14][::4] = 1e4 * (1.0 / 12.85) ** 2             # b = 1 km/s, pixels of 20
    args[15][::8] = 12000.0 / VELFAC
    args[7] = a * 4 * np.pi * 1e5 / HI_1215.lambda_cm     # a at b = 1 km/s
    args[13] = (args[13] * 1e6).astype(np.float32)
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    call = (nbins, kernel, VELFAC, dev(args[12]), dev(args[14]), [tuple(args[6:10])], [dev(args[13])])
    N.set_group_size(group)
    try:
        plan.keep_windows(True)
        got, handed = fp64_pairs(lambda: SP.tau(plan, *call)[0])
        weights = torch.exp(-1e-6 * got) + 0.5
        grads = SP.tau_adjoint(plan, *call, [weights])
        SP.set_fp64(True)
        SP.tau(plan, *call)
        want = SP.tau_adjoint(plan, *call, [weights])
    finally:
        SP.set_fp64(False)
        N.set_group_size(16)
    assert handed == 0
    assert_tau_close(got.cpu().numpy(), oracle.interpolate(*args), "wide supports")
    for x, y in zip((grads[0][0], grads[1], grads[2]), (want[0][0], want[1], want[2])):
        assert float((x - y).abs().max()) <= 1e-5 * float(y.abs().max())
    plan.close()


def replays_match(graph, outs, again):
    """Three replays, each against an eager call (into tensors of its own) in
    the shape that was captured."""
    for _ in range(3):
        for o in outs:
            o.fill_(-1.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for o, e in zip(outs, again()):
            assert torch.allclose(o, e, rtol=1e-12, atol=0)


def test_capture_in_another_launch_shape():
    """One uncaptured call with the same plan, lines and sizes is all that a
    capture needs, whatever lane-group width and wavefronts it then uses."""
    args = small_gas(4000, 900.0, 12, 256, 1, 0.1)
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    call = (dev(args[12]), dev(args[14]), [HI_1215], [dev(args[13])])
    outs = SP.tau(plan, 256, 1, VELFAC, *call)
    eager = outs[0].cpu().numpy().copy()
    graphs = []
    try:
        for group, waves in ((64, 4), (32, 2), (16, 8)):
            N.set_group_size(group)
            N.set_block_waves(waves)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                SP.tau(plan, 256, 1, VELFAC, *call, out=outs)
            graphs.append((group, waves, graph))
        for group, waves, graph in graphs:
            N.set_group_size(group)
            N.set_block_waves(waves)
            replays_match(graph, outs, lambda: SP.tau(plan, 256, 1, VELFAC, *call))
            assert_tau_close(outs[0].cpu().numpy(), eager, "captured")
    finally:
        N.set_group_size(16)
        N.set_block_waves(8)


def test_capture_after_autotune():
    """Many sightlines, of which the autotuner times every second one; the
    width it chose is captured after an eager call of another shape."""
    nlos, nbins = 33000, 16
    args = small_gas(300, 900.0, nlos, nbins, 1, 0.02)
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    call = (dev(args[12]), dev(args[14]), [HI_1215], [dev(args[13])])
    SP.autotune(plan, nbins, 1, VELFAC, *call)
    N.check(N.lib().fsamd_set_stats(1))                  # 4 wavefronts, with counters
    try:
        outs = SP.tau(plan, nbins, 1, VELFAC, *call)
    finally:
        N.check(N.lib().fsamd_set_stats(0))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        SP.tau(plan, nbins, 1, VELFAC, *call, out=outs)
    replays_match(graph, outs, lambda: SP.tau(plan, nbins, 1, VELFAC, *call))


def test_capture_of_column_density_after_tau():
    """The eager call with the same lines may be the other of the two."""
    args = small_gas(3000, 900.0, 9, 300, 1, 0.1)
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    vel, temp = dev(args[12]), dev(args[14])
    dens = [dev(args[13]), dev((args[13] * 2).astype(np.float32)), dev((args[13] * 3).astype(np.float32))]
    want = [o.clone() for o in SP.colden(plan, 300, 1, VELFAC, dens)]
    plan.close()
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    outs = [torch.empty((9, 300), dtype=torch.float64, device="cuda") for _ in dens]
    quad = (HI_1215.lambda_cm, HI_1215.gamma, HI_1215.fosc, HI_1215.amumass)
    SP.tau(plan, 300, 1, VELFAC, vel, temp, [quad] * 3, dens, out=outs)
    torch.cuda.synchronize()
    arr = SP._line_structs([quad] * 3, dens, outs)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        N.check(N.lib().fsamd_colden(plan.handle, 300, 1, VELFAC, SP._ptr(plan.pos), SP._ptr(plan.h), arr, 3,
                                     SP._stream()))
    replays_match(graph, outs, lambda: want)


# the longest rows of each lane-group width, and one pixel more
@pytest.mark.parametrize("group,most", [(16, 19536), (32, 19920), (64, 20112)])
def test_longest_adjoint_rows(group, most):
    args = small_gas(30, 700.0, 2, most, 1, 0.2)
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    plan.keep_windows(True)
    call = (dev(args[12]), dev(args[14]), [tuple(args[6:10])], [dev(args[13])])
    weights = dev(np.random.default_rng(4).standard_normal((2, most)))
    grads = []
    N.set_group_size(group)
    try:
        for fp64 in (False, True):
            SP.set_fp64(fp64)
            SP.tau(plan, most, 1, VELFAC, *call)
            gd, gt, gv = SP.tau_adjoint(plan, most, 1, VELFAC, *call, [weights])
            grads.append((gd[0], gt, gv))
        SP.set_fp64(False)
        t = SP.tau(plan, most + 1, 1, VELFAC, *call)[0]
        with pytest.raises(Exception, match="nbins too large"):
            SP.tau_adjoint(plan, most + 1, 1, VELFAC, *call, [t])
    finally:
        SP.set_fp64(False)
        N.set_group_size(16)
    for x, y in zip(*grads):
        assert float((x - y).abs().max()) <= 1e-5 * float(y.abs().max())
    plan.close()


# blocks of 4096 pixels, whose sums the host adds up where they are at most 32
@pytest.mark.parametrize("n", [4096, 4097, 32 * 4096, 32 * 4096 + 1, 1536 * 4096 + 1])
def test_mean_flux_of_few_and_many_blocks(n):
    import fluxstats as FS
    from fake_spectra_amd import fluxstatistics as GF
    t = np.exp(2.0 * np.random.default_rng(n).standard_normal(n))
    for target in (0.5, 0.95):
        got, ref = GF.mean_flux(dev(t), target, 1e-10), FS.mean_flux_scale(t, target, 1e-10)
        assert abs(got - ref) <= 1e-10 * ref      # the tolerance of the iteration


# rows of their own block, and short rows that share one from 1024 rows on, with a
# remainder and none
@pytest.mark.parametrize("nrow,ncol", [(1023, 5), (1024, 5), (1025, 50), (20001, 7), (40000, 3), (1600, 300)])
@pytest.mark.parametrize("sigma", [0.1, 1.04, 31.9])
def test_smoothing_of_rows_that_share_a_block(nrow, ncol, sigma):
    """A weighted mean of nw pixels: eps sqrt(nw) of the largest, with 4 ulp for
    the weights."""
    import fluxstats as FS
    from fake_spectra_amd import fluxstatistics as GF
    x = np.random.default_rng(ncol).random((nrow, ncol))
    dvbin = 8 / (2 * np.sqrt(2 * np.log(2))) / sigma
    got = GF.res_corr(dev(x), dvbin, 8).cpu().numpy()
    assert np.max(np.abs(got - FS.res_corr(x, dvbin, 8))) <= 2.3e-16 * (4 + np.sqrt(8 * sigma + 1)) * 2


# a negative cut that the first pixel lies within the guard band of, on either side
@pytest.mark.parametrize("off", [-1e-5, 1e-5, -1e-3, 1e-3])
def test_negative_cuts_of_negative_densities(oracle, off):
    """The walk ends at the first pixel below tautail: with a negative density
    (the difference of two fields) at once, or where it starts above, never."""
    args = list(small_gas(1, 900.0, 1, 200, 1, 0.02))
    args[12][:] = 0.0
    args[13] *= -1
    args[17] = args[11].astype(np.float64) + 1.0
    args[10] = -1e300
    whole = oracle.interpolate(*args)
    assert np.all(whole < 0)
    args[10] = float(whole.min()) * (1.0 + off)
    ref, got = oracle.interpolate(*args), SP._Particle_Interpolate(*args)
    assert np.count_nonzero(ref) < 200 if off < 0 else np.array_equal(ref, whole)
    assert np.array_equal(got == 0, ref == 0)
    assert np.max(np.abs(got - ref)) <= 1e-5 * np.max(np.abs(ref))
