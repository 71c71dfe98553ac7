"""The whole-iteration scan kernels against the plain FP64 scan.

The plain scan repeats the reference's arithmetic (tests/test_gpu_scan.py), so
it is the oracle here.  Sizes sit at the edges of what a lane holds: fewer
sites than lanes, exactly its resident sites, one more, an odd number of
streamed ones.  A trajectory keeps the plain scan's FIRE decisions when its
forces differ by rounding only (relative ~1e-14 a pair term, ~1e-12 A after a
height's iterations), so the step counts must be equal and positions within
1e-8 A, forces within 1e-8 of the largest force.
"""
import ctypes

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu


def _system(n, coul, rng, span=0.4):
    s = (abi.Site * max(n, 1))()
    r = 0.9 * np.sqrt(n) + 0.5
    for i in range(n):
        x, y = rng.uniform(-r, r, 2)
        s[i] = abi.Site(x + span / 2, y + span / 2, rng.normal(0, 0.1), abi.VDW_LJ, int(coul), 700.0, 1.1e6, 0.0,
                        -6.97 * rng.normal(0, 0.2) if coul else 0.0)
    d = abi.SystemDesc()
    d.n_sites, d.sites, d.force_grid, d.potential_grid = n, ctypes.cast(s, ctypes.POINTER(abi.Site)), -1, -1
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, 11077.0, 1.565e7, 0.0, 0.0, 0.72, 0.0)
    d.tip_dummy_d = 3.76
    return d, s


def _desc(nx, ny, nz, precision, lanes=0, integrator=1, minimiser=1, minterm=2, wpg=0, maxsteps=5000):
    d = abi.ScanDesc()
    for k, v in dict(nx=nx, ny=ny, nz=nz, dx=0.1, dy=0.1, dz=0.1, zhigh=9.0, minimiser=minimiser,
                     integrator=integrator, minterm=minterm, etol=0.01, ftol=0.01, dt=0.001, maxsteps=maxsteps,
                     precision=abi.PREC[precision], lanes_per_pixel=lanes, waves_per_group=wpg).items():
        setattr(d, k, v)
    return d


def _compare(ctx, systems, n, mk):
    ctx.set_systems(systems)
    ctx.scan(mk("plain64", 0))
    want = ctx.records(0, n)
    out = []
    for lanes in (0, 4, 8, 16, 32, 64):
        st = ctx.scan(mk("fast64", lanes))
        got = ctx.records(0, n)
        assert lanes == 0 or st["lanes_per_pixel"] == lanes
        np.testing.assert_array_equal(got["n_steps"], want["n_steps"])
        np.testing.assert_array_equal(got["flags"], want["flags"])
        for f in ("x", "y", "z"):
            np.testing.assert_array_equal(got[f], want[f])
        for f in ("rx", "ry", "rz"):
            assert np.abs(got[f] - want[f]).max() <= 1e-8
        big = max(np.abs(want[f]).max() for f in ("fx", "fy", "fz"))
        for f in ("fx", "fy", "fz", "e"):
            assert np.abs(got[f] - want[f]).max() <= 1e-8 * max(big, 1.0)
        out.append(st)
    return out


@pytest.mark.parametrize("coul", [False, True])
@pytest.mark.parametrize("n", [1, 7, 16, 33, 64, 129, 260])
def test_site_counts_and_lanes(gpu_ctx, n, coul):
    d, keep = _system(n, coul, np.random.default_rng(n))
    _compare(gpu_ctx, [d], 5 * 3 * 6, lambda p, g: _desc(5, 3, 6, p, g))


@pytest.mark.parametrize("minimiser,integrator,minterm", [(1, 0, 2), (1, 2, 2), (0, 1, 1), (1, 1, 0), (1, 1, 1)])
def test_minimisers(gpu_ctx, minimiser, integrator, minterm):
    d, keep = _system(37, True, np.random.default_rng(5))
    _compare(gpu_ctx, [d], 3 * 3 * 4, lambda p, g: _desc(3, 3, 4, p, g, integrator, minimiser, minterm))


@pytest.mark.parametrize("maxsteps", [1, 2, 12])
def test_heights_cut_short(gpu_ctx, maxsteps):
    d, keep = _system(40, True, np.random.default_rng(6))
    _compare(gpu_ctx, [d], 3 * 3 * 4, lambda p, g: _desc(3, 3, 4, p, g, maxsteps=maxsteps))


def test_dummy_coulomb_and_spring_length(gpu_ctx):
    d, keep = _system(40, True, np.random.default_rng(7))
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 1, 11077.0, 1.565e7, 0.0, -0.15, 0.72, 0.3)
    _compare(gpu_ctx, [d], 3 * 3 * 4, lambda p, g: _desc(3, 3, 4, p, g))


@pytest.mark.parametrize("wpg", [0, 1, 3, 8])
def test_batch_of_uneven_molecules(gpu_ctx, wpg):
    rng = np.random.default_rng(8)
    made = [_system(n, c, rng) for n, c in ((3, True), (90, False), (41, True), (160, True))]
    _compare(gpu_ctx, [d for d, _ in made], 4 * 5 * 5 * 4, lambda p, g: _desc(5, 5, 4, p, g, wpg=wpg))


@pytest.mark.parametrize("periodic,skew", [(False, False), (True, False), (True, True)])
def test_force_grid(gpu_ctx, periodic, skew):
    # a smooth field whose cells the scan crosses; on the periodic ones the
    # tip leaves the grid on every side
    n = (14, 12, 40) if not periodic else (9, 8, 40)
    basis = np.diag([0.1, 0.12, 0.09])
    if skew:
        basis[0, 1] = 0.03
    off = np.array([-0.4, -0.5, 2.0])
    I, J, K = np.meshgrid(*(np.arange(v) for v in n), indexing="ij")
    x, y, z = 2 * np.pi * I / n[0], 2 * np.pi * J / n[1], K * basis[2, 2] + off[2]
    amp = np.exp(-0.8 * (z - 2))
    fe = np.stack([0.4 * amp * np.sin(x), 0.4 * amp * np.cos(y), 1.5 * amp - 0.2, amp * (1 + 0.1 * np.cos(x + y))], -1)
    h = gpu_ctx.grid_upload(n, basis, off, fe.reshape(-1, 4), periodic)
    d, keep = _system(0, False, np.random.default_rng(1))
    d.force_grid = h
    gpu_ctx.set_systems([d])
    nx, ny, nz = (5, 4, 10)
    gpu_ctx.scan(_desc(nx, ny, nz, "plain64"))
    want = gpu_ctx.records(0, nx * ny * nz)
    st = gpu_ctx.scan(_desc(nx, ny, nz, "fast64"))
    got = gpu_ctx.records(0, nx * ny * nz)
    assert st["lanes_per_pixel"] == 8
    np.testing.assert_array_equal(got["n_steps"], want["n_steps"])
    np.testing.assert_array_equal(got["flags"], want["flags"])
    for f in ("fx", "fy", "fz", "rx", "ry", "rz", "e"):
        assert np.abs(got[f] - want[f]).max() <= 1e-8
    empty, keep2 = _system(0, False, np.random.default_rng(1))
    gpu_ctx.set_systems([empty])
    gpu_ctx.grid_free(h)


@pytest.mark.parametrize("potential", [False, True])
@pytest.mark.parametrize("n", [1, 9, 64, 130])
def test_periodic_images(gpu_ctx, n, potential):
    """3 x 3 images of an axis-aligned cell (nine reciprocals from one), with
    and without an external potential, and the general kernel for shifts that
    are no product; a periodic system's bars are those of the others."""
    rng = np.random.default_rng(n)
    cell = np.array([7.0, 6.0, 20.0])
    d, keep = _system(n, False, rng)
    h = -1
    if potential:
        g = (8, 6, 40)
        h = gpu_ctx.grid_upload(g, np.diag(cell / g), np.zeros(3), rng.normal(0, 0.05, (int(np.prod(g)), 4)), True)
    d.potential_grid, d.tip_pbc = h, 1
    for k in range(3):
        d.cell[4 * k] = cell[k]
    shifts = np.array([[i * cell[0], j * cell[1], 0.0] for i in (-1, 0, 1) for j in (-1, 0, 1)])
    for sh, product in ((shifts, True), (shifts + np.array([[0.0, 0.5 * (k // 3), 0.0] for k in range(9)]), False)):
        d.n_images, d.image_shifts = 9, sh.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        gpu_ctx.set_systems([d])
        gpu_ctx.scan(_desc(4, 3, 5, "plain64"))
        want = gpu_ctx.records(0, 60)
        for lanes in (0, 8, 16, 32, 64):
            gpu_ctx.scan(_desc(4, 3, 5, "fast64", lanes))
            got = gpu_ctx.records(0, 60)
            np.testing.assert_array_equal(got["n_steps"], want["n_steps"])
            np.testing.assert_array_equal(got["flags"], want["flags"])
            big = max(np.abs(want[f]).max() for f in ("fx", "fy", "fz"))
            for f in ("rx", "ry", "rz", "fx", "fy", "fz", "e"):
                assert np.abs(got[f] - want[f]).max() <= 1e-8 * max(big, 1.0)
    if potential:
        empty, keep2 = _system(0, False, rng)
        gpu_ctx.set_systems([empty])
        gpu_ctx.grid_free(h)


@pytest.mark.parametrize("coul", [False, True])
@pytest.mark.parametrize("n", [1, 5, 8, 16, 33, 64, 129, 260])
def test_flat_molecules(gpu_ctx, n, coul):
    """Sites of one height (their own kernels), off zero."""
    d, keep = _system(n, coul, np.random.default_rng(100 + n))
    for s in keep:
        s.z = -0.37
    _compare(gpu_ctx, [d], 5 * 3 * 6, lambda p, g: _desc(5, 3, 6, p, g))


def test_flat_molecules_of_several_heights_and_one_buckled(gpu_ctx):
    """A batch of flat molecules, each at its height, scans as flat; a buckled one among
    them takes it to the general kernels."""
    rng = np.random.default_rng(9)
    made = [_system(n, True, rng) for n in (30, 12, 50)]
    for k, (_, sites) in enumerate(made):
        for s in sites:
            s.z = 0.2 * k - 0.1
    _compare(gpu_ctx, [d for d, _ in made], 3 * 4 * 3 * 5, lambda p, g: _desc(4, 3, 5, p, g))
    made[1][1][3].z += 1e-3
    _compare(gpu_ctx, [d for d, _ in made], 3 * 4 * 3 * 5, lambda p, g: _desc(4, 3, 5, p, g))


@pytest.mark.parametrize("lanes", [4, 8])
def test_lanes_of_a_column_stay_together(gpu_ctx, tmp_path, lanes):
    """Relaxations of thousands of iterations along a ridge, where one rounding
    that differs between a column's lanes grows to 1e-4 A: a batch molecule at
    its full window against the plain scan."""
    from mechafm_amd import workloads as W
    sim = abi.Simulation(W.make_c3(str(tmp_path))[18].input_path, gpu_ctx)
    sim.run("plain64")
    want = sim.records()
    assert want["n_steps"].max() > 2000
    sim.run("fast64", lanes_per_pixel=lanes)
    got = sim.records()
    np.testing.assert_array_equal(got["n_steps"], want["n_steps"])
    for f in ("rx", "ry", "rz"):
        assert np.abs(got[f] - want[f]).max() <= 1e-8
    sim.close()
