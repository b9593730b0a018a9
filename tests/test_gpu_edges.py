"""Kernels at the sizes where their tiling can go wrong (edges of blocks,
strips and tiles, remainders, the smallest and largest of a range), against
the oracle."""
import numpy as np
import pytest

from fake_spectra_amd import spectra_priv as SP, synth
from fake_spectra_amd.lines import HI_1215
from gpu_util import assert_colden_close, assert_tau_close, dev

pytestmark = pytest.mark.gpu


def small_gas(n, box, nlos, nbins, kernel, hfrac, seed=3, line=HI_1215, compute_tau=True):
    """_Particle_Interpolate arguments for n particles of support about
    hfrac * box, two of them at one position, mixed axes."""
    rng = np.random.default_rng(seed)
    pos = (rng.random((n, 3)) * box).astype(np.float32)
    np.minimum(pos, np.nextafter(np.float32(box), np.float32(0)), out=pos)
    if n > 3:
        pos[n // 2] = pos[1]
    h = (hfrac * box * np.exp(0.2 * rng.standard_normal(n))).astype(np.float32)
    temp = (1e4 * np.exp(rng.standard_normal(n))).astype(np.float32)
    vel = (30.0 * rng.standard_normal((n, 3))).astype(np.float32)
    dens = np.exp(25.0 + rng.standard_normal(n)).astype(np.float32)
    axis = (1 + np.arange(nlos) % 3).astype(np.int32)
    cofm = rng.random((nlos, 3)) * box
    c = synth.Cosmology()
    none = np.zeros(1, dtype=np.float32)
    return (int(compute_tau), nbins, kernel, float(box), c.velfac(), c.atime, line.lambda_cm, line.gamma, line.fosc,
            line.amumass, 1e-7, pos, vel if compute_tau else none, dens, temp if compute_tau else none, h, axis, cofm)


# boxes of 2049, 2048, 2047 and 64 grid points 0.1 apart, one point, and rows
# of more particles than the candidates a block holds (every particle of the
# 850 of a row lies nearer than a block's stretch of points is long)
@pytest.mark.parametrize("box,n,nlos,hfrac", [(204.95, 400, 7, 0.3), (204.85, 400, 7, 0.3), (204.75, 300, 5, 0.3),
                                              (6.45, 60, 6, 0.4), (0.15, 5, 3, 0.4), (50.0, 3000, 4, 0.3),
                                              (1000.0, 3, 9, 0.4), (2000.0, 1500, 3, 0.15)])
def test_mesh_cells(oracle, box, n, nlos, hfrac):
    """The column density of kernel 2 is the overlap of a pixel with the
    particle's segment, so it pins the cells' ends."""
    for ct in (False, True):
        args = small_gas(n, box, nlos, 40, 2, hfrac, compute_tau=ct)
        ref = oracle.interpolate(*args)
        got = SP._Particle_Interpolate(*args)
        (assert_tau_close if ct else assert_colden_close)(got, ref, "mesh %g %d" % (box, n))


# mask words of 64 particles with every remainder kind, no, few and nearly all
# particles near a sightline, particles outside the box
@pytest.mark.parametrize("n,nlos,hfrac", [(1, 1, 0.4), (63, 2, 0.05), (64, 3, 0.3), (65, 1, 1e-4), (257, 700, 0.03),
                                          (4097, 50, 0.004), (1000, 1, 0.01)])
def test_near_lines(oracle, n, nlos, hfrac):
    args = small_gas(n, 1000.0, nlos, 8, 1, hfrac)
    box, pos, h, axis, cofm = args[3], args[11], args[15], args[16], args[17]
    if n > 64:
        pos[5] = [-3.0, 1001.0, 500.0]
    _, parts, _ = oracle.near_particles(box, pos, h, axis, cofm)
    got = SP._near_lines(box, pos, h, axis, cofm)
    assert got.dtype == np.int32 and np.array_equal(got, np.unique(parts))


# rows of fewer than 64, of 64, 65 and many pairs; supports of one or two pixels
# and of most of the row; every kernel; fields in one part, in several, and
# more than a launch takes; rows too long for two blocks and for LDS
@pytest.mark.parametrize("n,nlos,nbins,kernel,hfrac,fields", [
    (3, 4, 7, 1, 0.3, 1), (200, 3, 64, 3, 0.3, 5), (230, 5, 257, 0, 0.01, 2), (3000, 4, 1024, 1, 0.2, 5),
    (700, 3, 2048, 1, 0.02, 5), (700, 3, 4099, 3, 0.2, 4), (500, 2, 9001, 1, 0.1, 3), (300, 2, 20011, 1, 0.1, 2),
    (400, 3, 100, 9, 0.2, 11), (1, 1, 1, 1, 0.4, 1), (300, 4, 513, 2, 0.3, 3)])
def test_colden_fields(oracle, n, nlos, nbins, kernel, hfrac, fields):
    """Several fields of one plan, each against a call of its own; FP64
    throughout, so to rounding (a sum of up to ~1e4 positive terms)."""
    args = small_gas(n, 400.0, nlos, nbins, kernel, hfrac, compute_tau=False)
    pos, dens, h, axis, cofm = (args[i] for i in (11, 13, 15, 16, 17))
    rng = np.random.default_rng(9)
    all_dens = [dens] + [(dens * rng.random(n)).astype(np.float32) for _ in range(fields - 1)]
    plan = SP.Plan(args[3], dev(pos), dev(h), dev(axis), dev(cofm))
    if kernel == 2:
        plan.assign_cells()
    outs = SP.colden(plan, nbins, kernel, args[4], [dev(d) for d in all_dens])
    assert len(outs) == fields
    for d, o in zip(all_dens, outs):
        a = list(args)
        a[13] = d
        ref, got = oracle.interpolate(*a), o.cpu().numpy()
        assert np.array_equal(got == 0, ref == 0)
        assert np.max(np.abs(got - ref)) <= 1e-12 * max(ref.max(), 1e-300)


# damping parameters of 0, of cold and hot gas below 0.04, and above it; pixels
# of one midpoint and of many sub-samples; windows of one group step, several,
# and cut by half the row
@pytest.mark.parametrize("nbins,kernel,tscale,gscale", [(7, 1, 1.0, 1.0), (64, 3, 1e-4, 1.0), (300, 0, 1.0, 0.0),
                                                        (300, 1, 1.0, 40.0), (129, 1, 1e-3, 5.0), (1024, 1, 1.0, 1.0),
                                                        (200, 9, 1.0, 1e3)])
def test_fp64_walks(oracle, nbins, kernel, tscale, gscale):
    """Every pair on the FP64 path: the profile is good to ~1e-13 relative and
    the sums have positive terms, so tau to 1e-11."""
    args = list(small_gas(60, 1500.0, 3, nbins, kernel, 0.1))
    args[14] = (args[14] * tscale).astype(np.float32)
    args[7] *= gscale
    ref = oracle.interpolate(*args)
    SP.set_fp64(True)
    try:
        got = SP._Particle_Interpolate(*args)
    finally:
        SP.set_fp64(False)
    assert np.max(ref) > 0 and np.array_equal(got == 0, ref == 0)
    assert np.max(np.abs(got - ref) / np.maximum(ref, 1e-300)) <= 1e-11


# fewer sightlines than blocks (every row split, into one pair and into many),
# a row of no pairs, rows around the size of a part, rows too long for LDS, and
# rows of one to three pixels (windows of none and one a direction)
@pytest.mark.parametrize("n,nlos,nbins,hfrac", [(1, 1, 8, 0.4), (127, 2, 64, 0.5), (129, 1, 64, 0.5), (5000, 1, 300, 0.3),
                                                (400, 40, 100, 0.2), (3000, 2, 25000, 0.2), (3, 20, 50, 0.05),
                                                (5, 2, 1, 0.4), (5, 2, 2, 0.4), (40, 2, 3, 0.4)])
def test_split_rows(oracle, n, nlos, nbins, hfrac):
    """Rows cut into parts that add into the output: tau to the stated
    tolerance, column density to rounding, and forward and backward windows."""
    import torch
    from fake_spectra_amd import autograd as AG
    args = small_gas(n, 900.0, nlos, nbins, 1, hfrac)
    assert_tau_close(SP._Particle_Interpolate(*args), oracle.interpolate(*args), "split tau")
    cargs = small_gas(n, 900.0, nlos, nbins, 1, hfrac, compute_tau=False)
    ref, got = oracle.interpolate(*cargs), SP._Particle_Interpolate(*cargs)
    assert np.max(np.abs(got - ref)) <= 1e-12 * max(ref.max(), 1e-300)
    if nbins > 5000:
        return      # the adjoint keeps its rows in LDS
    # the gradient of the sum with respect to the densities is linear: sum over
    # particles of dens * grad equals the sum of tau (FP32 profile, 1e-5)
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    d = dev(args[13]).requires_grad_(True)
    tau = AG.tau_autograd(plan, nbins, 1, args[4], dev(args[12]), dev(args[14]), [HI_1215], [d])[0]
    total = tau.sum()
    if total.item() > 0:
        total.backward()
        assert float((d.grad.double() * d.detach().double()).sum()) == pytest.approx(total.item(), rel=1e-5)


# windows of no, one and many pixels, midpoints and many sub-samples, far wings
# (strong damping), light and full profiles side by side, rows beyond the
# adjoint's LDS and rows it refuses
@pytest.mark.parametrize("nbins,kernel,dscale,tscale,gscale", [(8, 1, 1.0, 1.0, 1.0), (64, 3, 1e3, 1e-2, 1.0),
                                                               (300, 0, 1e6, 1.0, 10.0), (1024, 1, 1e4, 1.0, 20.0),
                                                               (3200, 1, 1.0, 1.0, 1.0), (129, 1, 1e-9, 1.0, 1.0)])
def test_adjoint_against_fp64(nbins, kernel, dscale, tscale, gscale):
    """Gradients of sum(tau * weights) by the FP32 adjoint against the same
    windows by the FP64 one (fsamd_set_fp64, pinned to the torch reference):
    1e-5 of the largest of each gradient, the stated tolerance of tau."""
    import torch
    args = list(small_gas(150, 700.0, 3, nbins, kernel, 0.15))
    dens, temp = (args[13] * dscale).astype(np.float32), (args[14] * tscale).astype(np.float32)
    line = (args[6], args[7] * gscale, args[8], args[9])
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    plan.keep_windows(True)
    g = dev(np.random.default_rng(2).standard_normal((3, nbins)))
    out = {}
    for fp64 in (False, True):
        SP.set_fp64(fp64)
        try:
            SP.tau(plan, nbins, kernel, args[4], dev(args[12]), dev(temp), [line], [dev(dens)])
            gd, gT, gv = SP.tau_adjoint(plan, nbins, kernel, args[4], dev(args[12]), dev(temp), [line], [dev(dens)], [g])
        finally:
            SP.set_fp64(False)
        out[fp64] = [gd[0], gT, gv]
    for a, b in zip(out[False], out[True]):
        assert torch.isfinite(a).all()
        assert float((a - b).abs().max()) <= 1e-5 * float(b.abs().max())


def test_adjoint_refuses_long_rows():
    args = small_gas(20, 700.0, 1, 20000, 1, 0.2)
    plan = SP.Plan(args[3], dev(args[11]), dev(args[15]), dev(args[16]), dev(args[17]))
    plan.keep_windows(True)
    line, vel, temp, dens = args[6:10], dev(args[12]), dev(args[14]), dev(args[13])
    t = SP.tau(plan, 20000, 1, args[4], vel, temp, [line], [dens])[0]
    with pytest.raises(Exception, match="nbins too large"):
        SP.tau_adjoint(plan, 20000, 1, args[4], vel, temp, [line], [dens], [t])


# pixels of 1 to 129 sub-samples, around the counts where a lane group of 16, 32
# or 64 takes another number of rounds, pixels or none (FP64), in narrow and
# wide supports; rows of less than a step and of many
@pytest.mark.parametrize("group", [16, 32, 64])
@pytest.mark.parametrize("nbins,hfrac,kernel", [(200, 0.004, 1), (200, 0.05, 3), (9, 0.1, 1), (2048, 0.002, 0)])
def test_walks_of_all_sample_counts(oracle, group, nbins, hfrac, kernel):
    nm1 = np.array([0, 2, 4, 6, 8, 10, 14, 16, 20, 30, 32, 34, 62, 64, 66, 128] * 12)
    velfac = synth.Cosmology().velfac()
    args = list(small_gas(nm1.size, 20.0 * nbins / velfac, 4, nbins, kernel, hfrac))
    # a pixel is 20 km/s: b so that it has nm1 + 1 sub-samples (2 ceil(20 / b) + 1, one below b = 40)
    b = np.where(nm1 == 0, 50.0, 20.0 / (nm1 / 2 - 0.4))
    args[14] = (1e4 * (b / 12.85) ** 2).astype(np.float32)
    args[15] = np.maximum(args[15], np.float32(2.0 / velfac))
    args[16] = (1 + np.arange(4) % 3).astype(np.int32)
    rng = np.random.default_rng(7)
    args[17] = args[11][rng.integers(0, nm1.size, 4)].astype(np.float64) + 1e-3
    ref = oracle.interpolate(*args)
    from fake_spectra_amd import _native as N
    N.set_group_size(group)
    try:
        got = SP._Particle_Interpolate(*args)
    finally:
        N.set_group_size(16)
    assert np.max(ref) > 0
    assert_tau_close(got, ref, "sub-sample counts")


# supports that cross the box on either side of either axis, narrower than a
# cell, as wide as the box and wider; positions on its edges, outside it, far
# outside it and no numbers
@pytest.mark.parametrize("nlos", [1, 5, 40, 900])
@pytest.mark.parametrize("hfrac", [1e-4, 0.02, 0.3, 0.7, 3.0])
def test_windows_of_cells(oracle, nlos, hfrac):
    box = 1000.0
    args = small_gas(300, box, nlos, 8, 1, hfrac)
    pos, h, axis, cofm = args[11], args[15], args[16], args[17]
    edge = np.array([0.0, 0.3, np.nextafter(np.float32(box), np.float32(0)), 999.7, 500.0], dtype=np.float32)
    pos[:125] = np.stack(np.meshgrid(edge, edge, edge), -1).reshape(-1, 3)
    cofm[: nlos // 2] = np.where(cofm[: nlos // 2] < 500.0, 0.01 * cofm[: nlos // 2], 1000.0 - 0.01 * (1000.0 - cofm[: nlos // 2]))
    pos[130] = [-3.0, 1001.0, 500.0]
    pos[131] = [-2000.5, 0.1, 4000.5]
    pos[132] = [1e20, -1e20, 5.0]
    pos[133] = [np.nan, 10.0, 20.0]
    _, parts, _ = oracle.near_particles(box, pos, h, axis, cofm)
    assert np.array_equal(SP._near_lines(box, pos, h, axis, cofm), np.unique(parts))
    plan = SP.Plan(box, dev(pos), dev(h), dev(axis), dev(cofm))
    assert plan.npairs == len(parts)
    plan.close()


# grids of one block: fewer sightlines than its threads, as many, more; cells
# up to its limit (8192: 90 x 90 on one axis) and beyond; a sightline at
# infinity
@pytest.mark.parametrize("nlos,axes", [(1, 1), (2, 3), (1023, 3), (1025, 1), (4099, 3), (8100, 1), (8101, 1), (8400, 3)])
def test_grid_of_one_block(oracle, nlos, axes):
    box = 1000.0
    args = small_gas(200, box, nlos, 8, 1, 0.02)
    pos, h, axis, cofm = args[11], args[15], args[16], args[17]
    axis[:] = 1 + np.arange(nlos) % axes
    if nlos > 1000:
        cofm[17] = np.inf
        cofm[18, :] = cofm[19, :]
        cofm[20, :] = 0.0
        cofm[21, :] = box
    off, parts, _ = oracle.near_particles(box, pos, h, axis, cofm)
    plan = SP.Plan(box, dev(pos), dev(h), dev(axis), dev(cofm))
    got_off, got_parts = plan.pairs()
    assert np.array_equal(got_off.cpu().numpy(), off) and np.array_equal(got_parts.cpu().numpy(), parts)
    plan.close()


# offsets of one scan tile of 2048 entries, of several, of the 256 whose
# sums a block adds up itself, and of more; ends on and next to a tile's
@pytest.mark.parametrize("n", [1, 255, 2047, 2048, 2049, 524287, 524288, 524289, 1300000])
def test_offsets_of_all_scan_sizes(n):
    """One sightline that every second particle reaches: the neighbour list is
    those particles in order."""
    rng = np.random.default_rng(n)
    pos = (rng.random((n, 3)) * 1000.0).astype(np.float32)
    pos[:, 1:] = 500.0
    pos[1::2, 2] = 900.0
    h = np.full(n, 2.0, dtype=np.float32)
    plan = SP.Plan(1000.0, dev(pos), dev(h), dev(np.ones(1, dtype=np.int32)), dev(np.array([[0.0, 500.5, 500.5]])))
    off, parts = plan.pairs()
    want = np.arange(0, n, 2)
    assert off.cpu().tolist() == [0, want.size] and np.array_equal(parts.cpu().numpy(), want)
    plan.close()


# pairs of less than a sort tile (4096), one, one more, several and remainders;
# sightline ids of 1 to 17 bits, in one to three passes
@pytest.mark.parametrize("n,nlos", [(1, 1), (5, 2), (63, 65), (64, 64), (17, 241), (128, 64), (300, 257), (1, 4096), (1, 4097),
                                    (3, 70001), (2, 131072)])
def test_sorted_pairs_of_all_sizes(n, nlos):
    """Every particle reaches every sightline: each row holds all of them in
    order."""
    rng = np.random.default_rng(n)
    pos = (500.0 + rng.random((n, 3))).astype(np.float32)
    cofm = 500.0 + rng.random((nlos, 3))
    h = np.full(n, 300.0, dtype=np.float32)
    axis = (1 + np.arange(nlos) % 3).astype(np.int32)
    plan = SP.Plan(1000.0, dev(pos), dev(h), dev(axis), dev(cofm))
    off, parts = plan.pairs()
    assert np.array_equal(off.cpu().numpy(), n * np.arange(nlos + 1))
    assert np.array_equal(parts.cpu().numpy(), np.tile(np.arange(n), nlos))
    plan.close()
