"""Interaction lists of every shape on the GPU (System operators and flexible
scan) against the oracle: a few terms, one short of and past a wave's 64, one
to four waves, more rounds than a thread holds in registers, atoms with no
slot, one and more than eight, and lists whose state goes to HBM.

Tolerance: a term's values agree to 1e-9 (the device's acos / sin / atan / exp
against glibc's); a list that repeats terms r times sums r such differences,
and a step moves by dt times the force, less than it.
"""
import numpy as np
import pytest

from conftest import materialize
from mechafm_amd import abi
from oracle import oracle_flex as OF

pytestmark = pytest.mark.gpu

TOL = 1e-9


@pytest.fixture(scope="module")
def system(tmp_path_factory):
    return OF.flex_setup(materialize("fx_mini", str(tmp_path_factory.mktemp("fx_lists"))))


def _list(terms, size):
    """size terms of mixed kinds: the list's terms in a seeded order, repeated as
    often as it takes; the number of times."""
    order = np.random.default_rng(7).permutation(len(terms))
    reps = -(-size // len(terms))
    return terms[np.tile(order, reps)[:size]].copy(), reps


@pytest.mark.parametrize("size", [1, 2, 63, 64, 65, 128, 129, 257, 1100, 3000])
def test_list_sizes(gpu_ctx, system, size):
    fs = system
    terms, reps = _list(fs.terms, size)
    rng = np.random.default_rng(size)
    n = len(fs.fixed)
    pos = np.asarray(fs.base.system.pos)[None] + rng.normal(0, 0.02, (5, n, 3))
    pos[:, 1] = pos[:, 0] - [0.0, 0.0, fs.base.system.tip_dummy_d]
    vel, f0 = rng.normal(0, 0.05, (2, 5, n, 3))
    e0 = rng.normal(0, 0.5, (5, n))
    frc, ene = gpu_ctx.system_eval(terms, fs.fixed, pos, f0, e0)
    got = [gpu_ctx.system_step(terms, fs.fixed, i, 0.01, pos, vel, f0, e0) for i in range(3)]
    for s in range(len(pos)):
        f, e = f0[s].copy(), e0[s].copy()
        OF.system_op(terms, fs.fixed, "eval", pos[s].copy(), None, f, e)
        scale = max(1.0, np.abs(f).max(), np.abs(e).max())
        np.testing.assert_allclose(frc[s], f, rtol=0, atol=reps * TOL * scale)
        np.testing.assert_allclose(ene[s], e, rtol=0, atol=reps * TOL * scale)
        for i in range(3):
            want = [pos[s].copy(), vel[s].copy(), f0[s].copy(), e0[s].copy()]
            OF.system_op(terms, fs.fixed, "step", *want, integrator=i, dt=0.01)
            for g, w in zip(got[i], want):
                np.testing.assert_allclose(g[s], w, rtol=0, atol=reps * TOL * max(scale, np.abs(w).max()))


@pytest.mark.parametrize("size", [1, 64, 200, 900])
def test_scan_with_the_state_in_hbm_is_the_scan_in_lds(gpu_ctx, tmp_path, size):
    """Terms in registers and rows in LDS against both read from memory: the same
    records to the bit."""
    sim = abi.Simulation(materialize("fx_mini", str(tmp_path)), None)
    fx = sim.flex_system()
    i = sim.info()
    atom = fx["terms"]["atom"]
    ts = int(np.argmax((atom[:, 0] != 1) | (atom[:, 1] < 2)))       # the tip-surface terms come first
    terms = np.concatenate([fx["terms"][:ts], _list(fx["terms"][ts:], size)[0]])
    rec = []
    for opt in (0, abi.SCAN_STATE_IN_HBM):
        desc = sim.scan_desc("plain64", options=opt)
        desc.maxsteps = 40
        st = gpu_ctx.scan_flexible(fx["n_atoms"], fx["positions"], fx["fixed"], terms, desc, state_column=-1,
                                   tip_dummy_d=fx["tip_dummy_d"], cell=fx["cell"], offset=fx["offset"])
        rec.append(gpu_ctx.records(0, i["nx"] * i["ny"] * i["nz"]))
        assert st["total_steps"] == int(rec[-1]["n_steps"].sum())
    assert rec[0].tobytes() == rec[1].tobytes()
