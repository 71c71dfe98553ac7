"""Which kernels an FP64 scan takes by its number of columns: the whole-iteration ones
(at least four lanes a column), or past a line the general ones with one lane.
Records on both sides are those of the same columns scanned with lanes given:
the pair terms' rounding differs (relative ~1e-14), so values within 1e-8 and, over a
few iterations, equal step counts.
"""
import ctypes

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu


def _system(n, rng, cell=None):
    s = (abi.Site * max(n, 1))()
    for i in range(n):
        s[i] = abi.Site(*rng.uniform(0, 4, 2), rng.normal(0, 0.1), abi.VDW_LJ, int(cell is None), 700.0, 1.1e6, 0.0,
                        -6.97 * rng.normal(0, 0.2) if cell is None else 0.0)
    d = abi.SystemDesc()
    d.n_sites, d.sites, d.force_grid, d.potential_grid = n, ctypes.cast(s, ctypes.POINTER(abi.Site)), -1, -1
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, 11077.0, 1.565e7, 0.0, 0.0, 0.72, 0.0)
    d.tip_dummy_d = 3.76
    keep = [s]
    if cell is not None:
        sh = np.array([[i * cell, j * cell, 0.0] for i in (-1, 0, 1) for j in (-1, 0, 1)])
        d.n_images, d.image_shifts, d.tip_pbc = 9, sh.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 1
        for k, v in enumerate((cell, cell, 20.0)):
            d.cell[4 * k] = v
        keep.append(sh)
    return d, keep


def _desc(nx, lanes, integrator):
    d = abi.ScanDesc()
    for k, v in dict(nx=nx, ny=nx, nz=2, dx=4.0 / nx, dy=4.0 / nx, dz=0.1, zhigh=8.2, minimiser=1,
                     integrator=integrator, minterm=2, etol=0.01, ftol=0.01, dt=0.001, maxsteps=12,
                     precision=abi.PREC["fast64"], lanes_per_pixel=lanes, options=abi.SCAN_REPRODUCIBLE).items():
        setattr(d, k, v)
    return d


def _check(ctx, systems, nx, integrator, one_lane, other):
    n = len(systems) * nx * nx * 2
    ctx.set_systems(systems)
    st = ctx.scan(_desc(nx, 0, integrator))
    assert (st["lanes_per_pixel"] == 1) == one_lane
    got = ctx.records(0, n).copy()
    st = ctx.scan(_desc(nx, other, integrator))
    assert st["lanes_per_pixel"] == other
    want = ctx.records(0, n)
    for f in ("n_steps", "flags", "x", "y", "z"):
        np.testing.assert_array_equal(got[f], want[f])
    for f in ("rx", "ry", "rz", "fx", "fy", "fz", "e"):
        assert np.abs(got[f] - want[f]).max() <= 1e-8 * max(1.0, np.abs(want[f]).max())


@pytest.mark.parametrize("integrator,n,molecules,nx,one_lane",
                         [(1, 1, 1, 240, False), (1, 1, 1, 320, True), (1, 3, 8, 64, False), (1, 3, 32, 64, True),
                          (1, 40, 1, 400, False), (2, 1, 1, 256, False), (2, 1, 1, 420, True), (0, 4, 1, 128, False),
                          (0, 4, 1, 256, True)])
def test_sites(gpu_ctx, integrator, n, molecules, nx, one_lane):
    rng = np.random.default_rng(n)
    made = [_system(n, rng) for _ in range(molecules)]
    _check(gpu_ctx, [d for d, _ in made], nx, integrator, one_lane, 4 if one_lane else 1)


@pytest.mark.parametrize("sizes,nx,one_lane", [([6] * 63 + [200], 64, False), ([6] * 64, 64, True),
                                               ([6] * 60 + [100] * 4, 96, True)])
def test_uneven_molecules(gpu_ctx, sizes, nx, one_lane):
    rng = np.random.default_rng(len(sizes))
    made = [_system(n, rng) for n in sizes]
    _check(gpu_ctx, [d for d, _ in made], nx, 1, one_lane, 4 if one_lane else 1)


@pytest.mark.parametrize("integrator,n,nx,one_lane", [(1, 2, 160, False), (1, 2, 256, True), (1, 16, 256, False),
                                                      (0, 2, 128, False), (0, 2, 176, True)])
def test_images(gpu_ctx, integrator, n, nx, one_lane):
    d, keep = _system(n, np.random.default_rng(n), 4.0)
    _check(gpu_ctx, [d], nx, integrator, one_lane, 8 if one_lane else 1)


@pytest.mark.parametrize("integrator,nx,one_lane", [(1, 200, False), (1, 300, True), (0, 150, False), (0, 200, True)])
def test_force_grid(gpu_ctx, integrator, nx, one_lane):
    n = (50, 50, 40)
    x, y, z = (2 * np.pi * i / m for i, m in zip(np.meshgrid(*(np.arange(v) for v in n), indexing="ij"), n))
    amp = np.exp(-0.5 * z)
    fe = np.stack([0.4 * amp * np.sin(x), 0.4 * amp * np.cos(y), 1.5 * amp - 0.2, amp], -1)
    h = gpu_ctx.grid_upload(n, np.diag([0.1, 0.1, 0.1]), np.array([-0.5, -0.5, 2.0]), fe.reshape(-1, 4), True)
    d, keep = _system(0, np.random.default_rng(0))
    d.force_grid = h
    _check(gpu_ctx, [d], nx, integrator, one_lane, 8 if one_lane else 1)
    if not one_lane:              # the waves that the kernel's registers let a SIMD hold
        gpu_ctx.set_systems([d])
        assert gpu_ctx.scan(_desc(nx, 0, integrator))["waves_per_simd"] == (3 if integrator == 1 else 2)
    empty, keep2 = _system(0, np.random.default_rng(0))
    gpu_ctx.set_systems([empty])
    gpu_ctx.grid_free(h)
