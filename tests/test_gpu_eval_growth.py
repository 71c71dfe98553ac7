"""Tip-surface evaluations whose number of points grows from call to call: the pinned
memory they go through is allocated a few times, not by every call.  A call that
allocates takes ten times as long as one that does not, so the median of the
growing calls stays within three of the same calls repeated."""
import ctypes
import time

import numpy as np
import pytest

from mechafm_amd import abi

pytestmark = pytest.mark.gpu


def test_growing_calls_do_not_allocate_each_time():
    rng = np.random.default_rng(0)
    s = (abi.Site * 40)()
    for i in range(40):
        s[i] = abi.Site(*rng.uniform(0, 8, 2), 0.0, abi.VDW_LJ, 0, 700.0, 1.1e6, 0.0, 0.0)
    d = abi.SystemDesc()
    d.n_sites, d.sites, d.force_grid, d.potential_grid = 40, ctypes.cast(s, ctypes.POINTER(abi.Site)), -1, -1
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, 11077.0, 1.565e7, 0.0, 0.0, 0.72, 0.0)
    ctx = abi.Context(0)
    ctx.set_systems([d])
    pos = rng.uniform(2.0, 6.0, (8000, 3))
    want = ctx.eval_tip_surface(0, pos[:8000])
    ctx.close()
    ctx = abi.Context(0)
    ctx.set_systems([d])
    times = []
    for _ in range(2):                       # growing, then the same sizes again
        t = []
        for n in range(1100, 8000, 60):
            a = time.perf_counter()
            got = ctx.eval_tip_surface(0, pos[:n])
            t.append(time.perf_counter() - a)
            np.testing.assert_array_equal(got, want[:n])
        times.append(np.median(t))
    ctx.close()
    assert times[0] < 3 * times[1], times
