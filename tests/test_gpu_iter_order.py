"""The whole-iteration scan kernels: a pixel column's records do not depend on
its neighbours.

Two scans that share pixels deal them to other waves and other places in a
wave, so that other columns finish their heights beside them.  With reproducible
scans and the lanes given, a shared pixel's records must be the same bits: no
sum may be rounded one way beside a column that writes its record and another
way elsewhere.
"""
import ctypes

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu


def _desc(nx, ny, nz, lanes, integrator):
    d = abi.ScanDesc()
    for k, v in dict(nx=nx, ny=ny, nz=nz, dx=0.1, dy=0.1, dz=0.1, zhigh=9.0, minimiser=1, integrator=integrator,
                     minterm=2, etol=0.01, ftol=0.01, dt=0.001, maxsteps=5000, precision=abi.PREC["fast64"],
                     lanes_per_pixel=lanes, options=abi.SCAN_REPRODUCIBLE).items():
        setattr(d, k, v)
    return d


def _system(n, coul, flat, rng):
    s = (abi.Site * max(n, 1))()
    for i in range(n):
        s[i] = abi.Site(*rng.uniform(-4, 5, 2), 0.3 if flat else rng.normal(0, 0.1), abi.VDW_LJ, int(coul), 700.0,
                        1.1e6, 0.0, -6.97 * rng.normal(0, 0.2) if coul else 0.0)
    d = abi.SystemDesc()
    d.n_sites, d.sites, d.force_grid, d.potential_grid = n, ctypes.cast(s, ctypes.POINTER(abi.Site)), -1, -1
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, 11077.0, 1.565e7, 0.0, 0.0, 0.72, 0.0)
    d.tip_dummy_d = 3.76
    return d, s


def _check(ctx, d, lanes, integrator=1):
    nx, nz, most = 9, 6, 11
    ctx.set_systems([d])
    ctx.scan(_desc(nx, most, nz, lanes, integrator))
    whole = ctx.records(0, nx * most * nz).reshape(nx, most, nz)
    assert np.unique(whole["n_steps"]).size > 3
    for ny in (4, 7):
        ctx.scan(_desc(nx, ny, nz, lanes, integrator))
        part = ctx.records(0, nx * ny * nz).reshape(nx, ny, nz)
        for f in part.dtype.names:
            np.testing.assert_array_equal(part[f], whole[:, :ny][f], err_msg="%s, %d of %d rows" % (f, ny, most))


@pytest.mark.parametrize("lanes", [4, 8, 16, 32, 64])
@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("coul", [False, True])
def test_sites(gpu_ctx, coul, flat, lanes):
    d, keep = _system(83, coul, flat, np.random.default_rng(lanes))
    _check(gpu_ctx, d, lanes)


@pytest.mark.parametrize("integrator", [0, 2])
def test_other_integrators(gpu_ctx, integrator):
    d, keep = _system(41, True, False, np.random.default_rng(3))
    _check(gpu_ctx, d, 8, integrator)


@pytest.mark.parametrize("lanes", [8, 16, 64])
def test_images_with_a_potential(gpu_ctx, lanes):
    rng = np.random.default_rng(4)
    cell, g = np.array([9.0, 8.0, 20.0]), (8, 6, 40)
    d, keep = _system(50, False, False, rng)
    d.potential_grid = gpu_ctx.grid_upload(g, np.diag(cell / g), np.zeros(3), rng.normal(0, 0.05, (8 * 6 * 40, 4)), True)
    d.tip_pbc = 1
    for k in range(3):
        d.cell[4 * k] = cell[k]
    shifts = np.array([[i * cell[0], j * cell[1], 0.0] for i in (-1, 0, 1) for j in (-1, 0, 1)])
    d.n_images, d.image_shifts = 9, shifts.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    _check(gpu_ctx, d, lanes)
    empty, keep2 = _system(0, False, True, rng)
    gpu_ctx.set_systems([empty])
    gpu_ctx.grid_free(d.potential_grid)


def test_force_grid(gpu_ctx):
    n, h = (20, 22, 60), np.array([0.1, 0.1, 0.09])
    x, y, z = np.meshgrid(*(np.arange(v) * s for v, s in zip(n, h)), indexing="ij")
    amp = np.exp(-0.8 * z)
    fe = np.stack([0.4 * amp * np.sin(9 * x), 0.4 * amp * np.cos(7 * y), 1.5 * amp - 0.2, amp], -1).reshape(-1, 4)
    d, keep = _system(0, False, True, np.random.default_rng(1))
    d.force_grid = gpu_ctx.grid_upload(n, np.diag(h), np.array([-0.5, -0.5, 2.0]), fe, False)
    _check(gpu_ctx, d, 8)
    empty, keep2 = _system(0, False, True, np.random.default_rng(1))
    gpu_ctx.set_systems([empty])
    gpu_ctx.grid_free(d.force_grid)
