"""The whole-iteration scan kernels where numbers leave the ordinary range, against
the plain FP64 scan: what is finite there is finite and equal here.

Bars are the other scans' (tests/test_gpu_iter.py): equal step counts and flags,
values within 1e-8 of the plain scan's, relative where they are large.
"""
import ctypes

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu

D = 3.76              # tip below the dummy


def _system(sites, coul):
    """sites: positions; the first one is what a case is about."""
    s = (abi.Site * len(sites))()
    for i, p in enumerate(sites):
        s[i] = abi.Site(*p, abi.VDW_LJ, int(coul), 700.0, 1.1e6, 0.0, 0.4 if coul else 0.0)
    d = abi.SystemDesc()
    d.n_sites, d.sites, d.force_grid, d.potential_grid = len(sites), ctypes.cast(s, ctypes.POINTER(abi.Site)), -1, -1
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, 11077.0, 1.565e7, 0.0, 0.0, 0.72, 0.0)
    d.tip_dummy_d = D
    return d, s


def _desc(precision, lanes=0, nx=1, nz=1, dx=0.1, zhigh=D, maxsteps=5000, integrator=1):
    d = abi.ScanDesc()
    for k, v in dict(nx=nx, ny=nx, nz=nz, dx=dx, dy=dx, dz=0.1, zhigh=zhigh, minimiser=1, integrator=integrator,
                     minterm=2, etol=0.01, ftol=0.01, dt=0.001, maxsteps=maxsteps, precision=abi.PREC[precision],
                     lanes_per_pixel=lanes).items():
        setattr(d, k, v)
    return d


def _equal(ctx, system, n, lanes=(4, 8, 16, 32, 64), **kw):
    ctx.set_systems([system])
    ctx.scan(_desc("plain64", **kw))
    want = ctx.records(0, n)
    for g in lanes:
        ctx.scan(_desc("fast64", g, **kw))
        got = ctx.records(0, n)
        np.testing.assert_array_equal(got["n_steps"], want["n_steps"])
        np.testing.assert_array_equal(got["flags"], want["flags"])
        for f in ("rx", "ry", "rz", "fx", "fy", "fz", "e"):
            np.testing.assert_allclose(got[f], want[f], rtol=1e-8, atol=1e-8, err_msg="%s, %d lanes" % (f, g))
    return want


@pytest.mark.parametrize("coul", [False, True])
@pytest.mark.parametrize("flat", [False, True])
def test_tip_thrown_off_an_atom(gpu_ctx, coul, flat):
    """A tip that starts 1e-6 A above an atom: |v| |f| is past 1e154, |v| and |f| are not."""
    d, keep = _system([(0.0, 0.0, -1e-6), (0.0, 0.0, -1e-6 if flat else -2.0)], coul)
    want = _equal(gpu_ctx, d, 2, nz=2)
    assert np.isfinite(want["rz"]).all() and np.abs(want["rz"]).max() > 1e60


@pytest.mark.parametrize("coul", [False, True])
@pytest.mark.parametrize("flat", [False, True])
@pytest.mark.parametrize("integrator", [0, 1, 2])
def test_record_of_an_infinite_force(gpu_ctx, coul, flat, integrator):
    """A record taken 1.7e-24 A from an atom: its force is infinite, its energy is not."""
    a = 1e-24
    d, keep = _system([(a, a, a), (1.0, 1.0, a if flat else -2.0)], coul)
    want = _equal(gpu_ctx, d, 1, maxsteps=1, integrator=integrator)
    assert np.isinf(want["fz"]).all() and np.isfinite(want["e"]).all()


@pytest.mark.parametrize("coul", [False, True])
@pytest.mark.parametrize("height", [0.0, 1e4])
def test_scan_far_from_the_atoms(gpu_ctx, coul, height):
    """A column 10 000 A off, its tip at 10 000 A in all three coordinates: the lanes'
    padding is not there."""
    d, keep = _system([(0.0, 0.0, height), (1.5, 0.0, height), (0.0, 1.5, height)], coul)
    d.tip_dummy_d = 3.75
    _equal(gpu_ctx, d, 4, nx=2, dx=1e4, zhigh=10003.75)
    if not coul:
        shifts = np.array([[i * 30.0, j * 30.0, 0.0] for i in (-1, 0, 1) for j in (-1, 0, 1)])
        d.n_images, d.image_shifts = 9, shifts.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        _equal(gpu_ctx, d, 4, lanes=(8, 16, 32, 64), nx=2, dx=1e4, zhigh=10003.75)
