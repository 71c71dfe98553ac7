"""Tip-surface evaluations on both sides of the numbers of points where the lanes a
point change: a point's force and energy do not depend on them, bit for bit."""
import ctypes

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sites", [7, 63, 64])
def test_a_point_does_not_depend_on_the_number_of_points(gpu_ctx, sites):
    rng = np.random.default_rng(sites)
    s = (abi.Site * sites)()
    for i in range(sites):
        s[i] = abi.Site(*rng.uniform(0, 8, 2), rng.normal(0, 0.1), abi.VDW_LJ, i % 2, 700.0, 1.1e6, 0.0, 0.3)
    d = abi.SystemDesc()
    d.n_sites, d.sites, d.force_grid, d.potential_grid = sites, ctypes.cast(s, ctypes.POINTER(abi.Site)), -1, -1
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, 11077.0, 1.565e7, 0.0, 0.0, 0.72, 0.0)
    gpu_ctx.set_systems([d])
    pos = rng.uniform(2.0, 6.0, (90001, 3))
    want = np.concatenate([gpu_ctx.eval_tip_surface(0, pos[a:a + 4000]) for a in range(0, len(pos), 4000)])
    for n in (4096, 4097, 8192, 8193, 40000, 40001, 90000, 90001):
        np.testing.assert_array_equal(gpu_ctx.eval_tip_surface(0, pos[:n]), want[:n], err_msg=str(n))
