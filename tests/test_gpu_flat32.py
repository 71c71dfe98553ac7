"""The FP32 scan of flat molecules (sites of one height) against the general
FP32 kernel.

The flat kernel forms dz and dz^2 once instead of site by site and changes no
other operation, so its records are the general kernel's bit for bit.  A batch
takes the general kernel as soon as one of its molecules is buckled: the flat
molecule's records from a batch of its own and from one beside a buckled
molecule must be the same.  Sizes sit at the edges of a lane's register blocks
(6 Lennard-Jones or 4 Morse sites) and of its remainder; summation order is
fixed (reproducible scans, lanes given).
"""
import ctypes

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu


def _system(n, kinds, z, rng):
    """n sites at height z (one of them off it when z is None); kinds: the
    (vdw, charged) pairs the sites go through in turn."""
    s = (abi.Site * n)()
    r = 0.9 * np.sqrt(n) + 0.5
    for i in range(n):
        vdw, charged = kinds[i % len(kinds)]
        p = (700.0, 1.1e6, 0.0) if vdw == abi.VDW_LJ else (0.3, 1.6, 3.4)
        s[i] = abi.Site(*rng.uniform(-r, r, 2), 0.05 * i if z is None else z, vdw, int(charged), *p,
                        -6.97 * rng.normal(0, 0.2) if charged else 0.0)
    d = abi.SystemDesc()
    d.n_sites, d.sites, d.force_grid, d.potential_grid = n, ctypes.cast(s, ctypes.POINTER(abi.Site)), -1, -1
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, 11077.0, 1.565e7, 0.0, 0.0, 0.72, 0.0)
    d.tip_dummy_d = 3.76
    return d, s


@pytest.mark.parametrize("kinds", [[(abi.VDW_LJ, True)], [(abi.VDW_LJ, False)],
                                   [(abi.VDW_LJ, True), (abi.VDW_LJ, False), (abi.VDW_MORSE, True),
                                    (abi.VDW_MORSE, False)]], ids=["charged", "plain", "mixed"])
@pytest.mark.parametrize("lanes", [1, 2, 8, 64])
def test_flat_equals_general(gpu_ctx, lanes, kinds):
    d = abi.ScanDesc()
    for k, v in dict(nx=5, ny=3, nz=4, dx=0.1, dy=0.1, dz=0.1, zhigh=9.0, minimiser=1, integrator=1, minterm=2,
                     etol=0.01, ftol=0.01, dt=0.001, maxsteps=5000, precision=abi.PREC["fast32"],
                     lanes_per_pixel=lanes, options=abi.SCAN_REPRODUCIBLE).items():
        setattr(d, k, v)
    rng = np.random.default_rng(lanes)
    made = [_system(n, kinds, z, rng) for n, z in ((1, 0.4), (6 * lanes, -0.37), (6 * lanes + 1, 0.0),
                                                   (13 * lanes - 1, 1.25))]
    buckled = _system(9, kinds, None, rng)
    n = len(made) * 5 * 3 * 4
    gpu_ctx.set_systems([x for x, _ in made])
    gpu_ctx.scan(d)
    flat = gpu_ctx.records(0, n).copy()
    gpu_ctx.set_systems([x for x, _ in made] + [buckled[0]])
    gpu_ctx.scan(d)
    general = gpu_ctx.records(0, n)
    assert np.abs(flat["fz"]).max() > 0
    for f in flat.dtype.names:
        np.testing.assert_array_equal(flat[f], general[f], err_msg=f)
