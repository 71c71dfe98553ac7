"""The smallest flexible systems, two and three atoms: the tip's ordered sum runs
ahead of its list to the end of the block's state.  System operators against the
oracle (a term's values to 1e-9, the bar of the larger lists), the flexible scan
in LDS against the same in memory, bit for bit.
"""
import numpy as np
import pytest

from mechafm_amd import abi
from oracle import oracle_flex as OF

pytestmark = pytest.mark.gpu


def _terms(n, reps):
    rows = [(abi.FX_LJ, (1, 2), (700.0, 1.1e6))] * reps if n > 2 else []
    rows += [(abi.FX_LJ, (0, 1), (11077.0, 1.565e7)), (abi.FX_TIP_HARMONIC, (1, 0), (0.72, 0.1)),
             (abi.FX_XY_HARMONIC, (1,), (0.3, 0.05, -0.04))] * reps
    if n > 2:
        rows += [(abi.FX_XY_HARMONIC, (2,), (2.0, 0.1, 0.1)), (abi.FX_SUBSTRATE, (2,), (3.0, 0.4, 0.1, -3.0, 8.0, 3.0))]
    t = np.zeros(len(rows), dtype=abi.FLEX_TERM_DTYPE)
    for k, (kind, atoms, p) in enumerate(rows):
        t[k]["kind"] = kind
        t[k]["atom"][:len(atoms)] = atoms
        t[k]["p"][:len(p)] = p
    return t


@pytest.mark.parametrize("n", [2, 3])
@pytest.mark.parametrize("reps", [0, 1, 5, 6, 16])
def test_operators(gpu_ctx, n, reps):
    terms = _terms(n, reps)
    fixed = np.array([1, 0, 0], dtype=np.int32)[:n]
    rng = np.random.default_rng(reps)
    base = np.array([[0.0, 0.0, 7.5], [0.0, 0.0, 3.74], [0.1, 0.0, 0.0]])[:n]
    pos = base[None] + rng.normal(0, 0.02, (4, n, 3))
    vel, f0 = rng.normal(0, 0.05, (2, 4, n, 3))
    e0 = rng.normal(0, 0.5, (4, n))
    frc, ene = gpu_ctx.system_eval(terms, fixed, pos, f0, e0)
    got = [gpu_ctx.system_step(terms, fixed, i, 0.01, pos, vel, f0, e0) for i in range(3)]
    tol = 1e-9 * max(reps, 1)
    for s in range(len(pos)):
        f, e = f0[s].copy(), e0[s].copy()
        OF.system_op(terms, fixed, "eval", pos[s].copy(), None, f, e)
        np.testing.assert_allclose(frc[s], f, rtol=tol, atol=tol)
        np.testing.assert_allclose(ene[s], e, rtol=tol, atol=tol)
        for i in range(3):
            want = [pos[s].copy(), vel[s].copy(), f0[s].copy(), e0[s].copy()]
            OF.system_op(terms, fixed, "step", *want, integrator=i, dt=0.01)
            for g, w in zip(got[i], want):
                np.testing.assert_allclose(g[s], w, rtol=tol, atol=tol)
    for integrator in range(3):
        p, v, f, e, steps = gpu_ctx.system_minimise(terms, fixed, pos, vel, energies=e0, integrator=integrator,
                                                    maxsteps=6, etol=0.0, ftol=0.0, minterm=2)
        assert (steps == 6).all() and np.isfinite(p).all() and np.isfinite(e).all()


@pytest.mark.parametrize("n", [2, 3])
@pytest.mark.parametrize("reps", [0, 1, 6, 16])
@pytest.mark.parametrize("integrator", [1, 2])
def test_scan_in_lds_is_the_scan_in_memory(gpu_ctx, n, reps, integrator):
    terms = _terms(n, reps)
    rec = []
    for opt in (0, abi.SCAN_STATE_IN_HBM):
        d = abi.ScanDesc()
        for k, v in dict(nx=3, ny=2, nz=3, dx=0.1, dy=0.1, dz=0.1, zhigh=7.5, minimiser=1, integrator=integrator,
                         minterm=2, etol=0.01, ftol=0.01, dt=0.001, maxsteps=300, precision=abi.PREC["plain64"],
                         options=opt).items():
            setattr(d, k, v)
        gpu_ctx.scan_flexible(n, np.array([[0, 0, 7.5], [0, 0, 3.74], [0.1, 0, 0]])[:n], [1, 0, 0][:n], terms, d,
                              tip_dummy_d=3.76)
        rec.append(gpu_ctx.records(0, 18).copy())
    assert rec[0].tobytes() == rec[1].tobytes()
    assert np.isfinite(rec[0]["rz"]).all()
