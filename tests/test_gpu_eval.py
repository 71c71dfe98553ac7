"""The tip-surface operator's ways through the chip give the same bits: 64 lanes
a point from pinned memory, 16 lanes from device memory and a lane a point, at
their edges in points and sites, for every kind of site, over periodic images,
on top of an external grid and off its edge.  (Against the oracle the operator
is tested elsewhere; 131073 points go one lane a point.)"""
import ctypes

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu

ONE_LANE = 131073


def _system(rng, sites, kind, images=1):
    arr = (abi.Site * sites)()
    for i in range(sites):
        morse = kind == "morse" or (kind == "mixed" and i % 3 == 1)
        p = (0.01, 1.8, 3.4) if morse else (5.0 + i, 4.0e3, 0.0)
        arr[i] = abi.Site(*rng.uniform(-4, 4, 2), rng.normal(0, 0.2), abi.VDW_MORSE if morse else abi.VDW_LJ,
                          int(kind != "bare" and i % 4 != 2), *p, rng.normal(0, 3.0))
    d = abi.SystemDesc()
    d.n_sites, d.sites = sites, ctypes.cast(arr, ctypes.POINTER(abi.Site))
    d.force_grid = d.potential_grid = -1
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, 300.0, 1e5, 0.0, 0.0, 0.1, 0.0)
    d.tip_dummy_d = 3.0
    shifts = np.array([[9.0 * k, -9.0 * k, 0.0] for k in range(images)])
    if images > 1:
        d.n_images, d.image_shifts = images, shifts.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    return d, (arr, shifts)


def _same(ctx, pos, counts):
    ref = ctx.eval_tip_surface(0, np.resize(pos, (ONE_LANE, 3)))
    for n in counts:
        got = ctx.eval_tip_surface(0, pos[:n])
        assert got.tobytes() == ref[:n].tobytes(), f"{n} points"


@pytest.mark.parametrize("kind", ["bare", "lj", "morse", "mixed"])
@pytest.mark.parametrize("sites", [1, 8, 15, 16, 17, 63, 64, 65, 130])
def test_split_sums_are_the_serial_sums(gpu_ctx, sites, kind):
    rng = np.random.default_rng(sites)
    d, _keep = _system(rng, sites, kind)
    gpu_ctx.set_systems([d])
    pos = rng.uniform([-5, -5, 2.5], [5, 5, 7], (9000, 3))
    _same(gpu_ctx, pos, [1, 3, 4, 5, 255, 4096, 4097, 8192, 8193, 9000])


@pytest.mark.parametrize("images", [2, 9])
def test_images(gpu_ctx, images):
    rng = np.random.default_rng(images)
    d, _keep = _system(rng, 70, "mixed", images)
    gpu_ctx.set_systems([d])
    _same(gpu_ctx, rng.uniform([-5, -5, 2.5], [5, 5, 7], (4100, 3)), [1, 100, 4096, 4100])


def test_external_grid_and_its_edge(gpu_ctx):
    rng = np.random.default_rng(0)
    n = (12, 10, 9)
    h = gpu_ctx.grid_upload(n, np.diag([1.0, 1.0, 1.0]), np.array([-6.0, -5.0, 0.0]), rng.normal(size=(*n, 4)), False)
    d, _keep = _system(rng, 40, "lj")
    d.potential_grid = h
    gpu_ctx.set_systems([d])
    pos = rng.uniform([-4, -4, 2.5], [4, 3, 7], (5000, 3))
    _same(gpu_ctx, pos, [1, 100, 4096, 4097, 5000])
    for m in (1, 10, 5000, ONE_LANE):
        bad = np.resize(pos, (m, 3)).copy()
        bad[m // 2, 0] = 50.0
        with pytest.raises(abi.MafmError, match="past the force grid"):
            gpu_ctx.eval_tip_surface(0, bad)
    _same(gpu_ctx, pos, [10])
    d2, _keep2 = _system(rng, 4, "lj")
    gpu_ctx.set_systems([d2])
    gpu_ctx.grid_free(h)
