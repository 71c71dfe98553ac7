"""Workloads of the framework for timing and for comparing two builds.

Each case is a dict of plain values; ``prepare`` makes what a program has in
hand before the call (systems, grids, input files, context), ``run`` is one
call through the public entry points with its whole result.  The kinds:

  forces     tip-surface forces at given tip positions: the smallest call,
             what a calculator asks for between its own steps
  scan       force curves and images of isolated molecules, records on the
             host (mafm_scan + mafm_records); with ``deltaf`` the
             frequency-shift images as well
  batch      many molecules in one launch, records in the caller's device
             memory (mafm_scan_noalloc): screening and data-set generation
  rigidgrid  jobs with ``rigidgrid on``, one after the other: sample the
             force grid, scan through it, free the grid of the job before
  slab       periodic surface with nine images and an external potential
  gradient   one step of a fit: image, loss, gradients of every parameter
  potential  external potential from a cube: FFT convolution and spectral
             gradient, the grid back on the host
  flexible   the whole surface relaxing under the tip, from a job's files
  relax      many copies of a flexible system minimised at once

Scan geometry, FIRE settings, pair parameters and sizes are those of the
workloads in mechafm_amd.workloads (flake, 40-atom, 64-molecule, slab,
150-atom and flexible jobs); every seed gives other atoms, charges or states.
"""
import ctypes
import math
import os
import sys
import tempfile

import numpy as np
import torch

from mechafm_amd import abi, workloads
from mechafm_amd.adjoint import ScanModel

LIST = [
    # a calculator's single query of a tip-surface force field
    dict(name="forces", kind="forces", atoms=150, points=1000, vdw="lj"),
    # one force-distance curve over the 96-atom flake: one pixel column
    dict(name="curve", kind="scan", shape="flake", atoms=96, nx=1, ny=1, nz=41, coulomb=False, minimiser=1,
         integrator=1, deltaf=False),
    # the 96-atom flake's image: every height, and its frequency-shift images
    dict(name="flake", kind="scan", shape="flake", atoms=96, nx=101, ny=101, nz=41, coulomb=False, minimiser=1,
         integrator=1, deltaf=True),
    # a charged, buckled molecule with the RK4 integrator
    dict(name="flake_rk4", kind="scan", shape="buckled", atoms=131, nx=33, ny=33, nz=41, coulomb=True, minimiser=1,
         integrator=2, deltaf=False),
    # 40 atoms, Morse + Coulomb, sampled on a force grid of half the scan's spacing
    dict(name="rigidgrid", kind="rigidgrid", atoms=40, nx=128, ny=128, nz=36),
    # 64 planar molecules of 20 to 400 atoms in one launch, FP64 pair terms
    dict(name="batch", kind="batch", precision="fast64", molecules=64, nmin=20, nmax=400, nx=64, ny=64, nz=40),
    # the same kind of batch with FP32 pair terms, fewer molecules
    dict(name="batch_fp32", kind="batch", precision="fast32", molecules=20, nmin=20, nmax=400, nx=64, ny=64, nz=40),
    # 2000 atoms in a 40 x 40 A cell with its images and an external potential
    dict(name="slab", kind="slab", atoms=2000, cell=40.0, n_grid=160, nx=64, ny=64, nz=40),
    # a 150-atom molecule's image and the gradient of an image loss
    dict(name="gradient", kind="gradient", area=12.75, zlow=7.05),
    # the external potential of a 160 x 160 x 80 cube
    dict(name="potential", kind="potential", n0=160, n1=160, n2=80),
    # the 72-atom graphene job of the examples with every atom free to relax
    dict(name="flexible", kind="flexible", ax=20.0, ay=15.0, zlow=6.0),
    # 300 perturbed copies of a flexible flake with a tip above it
    dict(name="relax", kind="relax", states=300),
]


def listed():
    return [dict(c) for c in LIST]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forces", "scan", "scan", "scan", "batch", "batch", "rigidgrid", "slab", "gradient",
                       "potential", "flexible", "relax"])
    if kind == "forces":
        return dict(kind=kind, atoms=_log(rng, 20, 400), points=_log(rng, 1, 200000), vdw=rng.choice(["lj", "morse"]))
    if kind == "scan":
        integrator = rng.choice([1, 1, 1, 0, 2])
        most = 128 if integrator == 1 else 40
        n = [_log(rng, 1, most), _log(rng, 1, most)]
        return dict(kind=kind, shape=rng.choice(["flake", "buckled"]), atoms=_log(rng, 20, 400), nx=n[0], ny=n[1],
                    nz=rng.randint(20, 41), coulomb=rng.random() < 0.7, minimiser=1, integrator=integrator,
                    deltaf=rng.random() < 0.3)
    if kind == "batch":
        nmin = _log(rng, 20, 100)
        return dict(kind=kind, precision=rng.choice(["fast64", "fast64", "fast32"]), molecules=_log(rng, 2, 40),
                    nmin=nmin, nmax=rng.randint(nmin, 400), nx=rng.randint(16, 64), ny=rng.randint(16, 64),
                    nz=rng.randint(20, 40))
    if kind == "rigidgrid":
        return dict(kind=kind, atoms=_log(rng, 12, 120), nx=_log(rng, 16, 128), ny=_log(rng, 16, 128),
                    nz=rng.randint(18, 34))
    if kind == "slab":
        cell = rng.choice([12.0, 20.0, 28.0, 40.0])
        return dict(kind=kind, atoms=int(cell * cell * 1.25), cell=cell, n_grid=int(4 * cell), nx=rng.randint(8, 64),
                    ny=rng.randint(8, 64), nz=rng.randint(10, 40))
    if kind == "gradient":
        return dict(kind=kind, area=round(rng.uniform(2.0, 12.7), 2), zlow=round(rng.uniform(7.1, 9.0), 2))
    if kind == "potential":
        a, b, c = (rng.choice([24, 40, 54, 64, 75, 80, 96, 110, 128, 156, 160]) for _ in range(3))
        return dict(kind=kind, n0=a, n1=b, n2=c)
    if kind == "flexible":
        return dict(kind=kind, ax=round(rng.uniform(1.0, 20.0), 1), ay=round(rng.uniform(1.0, 15.0), 1),
                    zlow=round(rng.uniform(6.0, 9.0), 1))
    return dict(kind="relax", states=_log(rng, 1, 400))


# ---------------------------------------------------------------- systems
QBASE = 332.06371                       # kcal/mol A / e^2
TIP, DUMMY = "O", "X"
ATOMS = workloads.BASE_ATOMS            # eps, sigma, mass, charge
SCAN = dict(dx=0.1, dy=0.1, dz=0.1, zhigh=10.0, minterm=2, etol=0.01, ftol=0.01, dt=0.001, maxsteps=5000)


def _mix(a, b):
    eps, sig = math.sqrt(ATOMS[a][0] * ATOMS[b][0]), 0.5 * (ATOMS[a][1] + ATOMS[b][1])
    return 4 * eps * sig ** 6, 4 * eps * sig ** 12, eps, sig


def _molecule(rng, n, span, shape):
    """n atoms of a honeycomb patch around the middle of the scanned area:
    elements, charges and, for "flake", only carbons; planar unless "buckled".
    A patch is laid anew for every seed (place, rotation, small displacements)."""
    c = 1.42
    k = int(math.sqrt(n)) + 4
    u, v = np.meshgrid(np.arange(-k, k + 1), np.arange(-k, k + 1), indexing="ij")
    a = np.stack([math.sqrt(3) * c * (u + 0.5 * v), 1.5 * c * v], -1).reshape(-1, 2)
    xy = np.concatenate([a, a + np.array([0.0, c])]) + rng.uniform(-0.7, 0.7, 2)
    xy = xy[np.argsort((xy ** 2).sum(1), kind="stable")[:n]]
    t = rng.uniform(0, 2 * math.pi)
    xy = xy @ np.array([[math.cos(t), -math.sin(t)], [math.sin(t), math.cos(t)]])
    pos = np.zeros((n, 3))
    pos[:, :2] = xy + rng.uniform(-0.04, 0.04, (n, 2)) + 0.5 * np.asarray(span)
    if shape == "buckled":
        pos[:, 2] = rng.normal(0.0, 0.15, n)
    types = ["C"] * n if shape == "flake" else list(rng.choice(["C", "N", "O", "H"], size=n, p=[0.5, 0.15, 0.10, 0.25]))
    q = rng.normal(0.0, 0.2, n)
    return types, pos, q - q.mean()


def _constants(types, q, coulomb, vdw):
    """Per atom: p0, p1, p2 of its pair term with the tip, and its Coulomb prefactor."""
    p = np.zeros((len(types), 3))
    for i, t in enumerate(types):
        es6, es12, eps, sig = _mix(TIP, t)
        p[i] = (es6, es12, 0.0) if vdw == "lj" else (eps, 1.8, sig * 2 ** (1 / 6))
    qq = QBASE * ATOMS[TIP][3] * q if coulomb else np.zeros(len(types))
    return p, qq


def _system(types, pos, q, coulomb, vdw, images=None, cell=None):
    """mafm_system_desc of one molecule; keep the returned list alive beside it."""
    p, qq = _constants(types, q, coulomb, vdw)
    s = (abi.Site * len(types))()
    kind = abi.VDW_LJ if vdw == "lj" else abi.VDW_MORSE
    for i in range(len(types)):
        s[i] = abi.Site(pos[i, 0], pos[i, 1], pos[i, 2], kind, int(coulomb), p[i, 0], p[i, 1], p[i, 2], qq[i])
    d = abi.SystemDesc()
    d.n_sites, d.sites = len(types), ctypes.cast(s, ctypes.POINTER(abi.Site))
    d.force_grid = d.potential_grid = -1
    es6, es12, _, sig = _mix(TIP, DUMMY)
    d.tip_dummy = abi.TipDummy(abi.VDW_LJ, 0, es6, es12, 0.0, 0.0, workloads.HARM[0], workloads.HARM[1])
    d.tip_dummy_d = sig * 2 ** (1 / 6)
    keep = [s]
    if images is not None:
        im = np.ascontiguousarray(images, dtype=np.float64)
        d.n_images, d.image_shifts, d.tip_pbc = len(im), im.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), 1
        for k, v in enumerate(np.diag(cell).ravel()):
            d.cell[k] = v
        keep.append(im)
    return d, keep


def _scan_desc(c, precision="fast64", **kw):
    d = abi.ScanDesc()
    for k, v in dict(SCAN, nx=c["nx"], ny=c["ny"], nz=c["nz"], minimiser=c.get("minimiser", 1),
                     integrator=c.get("integrator", 1), precision=abi.PREC[precision], **kw).items():
        setattr(d, k, v)
    return d


def _span(c):
    return [(c["nx"] - 1) * SCAN["dx"], (c["ny"] - 1) * SCAN["dy"]]


def _fields(rec):
    return {k: rec[k] for k in rec.dtype.names}


def _tip_points(c, rng):
    """Tip positions 2.6 to 6 A above a molecule."""
    r = 0.9 * math.sqrt(c["atoms"])
    return np.stack([rng.uniform(-r, r, c["points"]), rng.uniform(-r, r, c["points"]),
                     rng.uniform(2.6, 6.0, c["points"])], 1)


def _cube(c, rng):
    """Potential of random charges (energy units, tens of kcal/mol/e) on the
    grid: white noise damped as a Gaussian of 0.6 A and by 1/k^2 in k space."""
    n = (c["n0"], c["n1"], c["n2"])
    g = torch.Generator(device="cuda").manual_seed(int(rng.integers(1 << 30)))
    x = torch.fft.fftn(torch.randn(n, dtype=torch.float64, device="cuda", generator=g))
    k = [2 * math.pi * torch.fft.fftfreq(m, d=0.25, dtype=torch.float64, device="cuda") for m in n]
    k2 = k[0][:, None, None] ** 2 + k[1][None, :, None] ** 2 + k[2][None, None, :] ** 2
    k2[0, 0, 0] = 1.0
    f = torch.exp(-0.5 * 0.36 * k2) / k2
    f[0, 0, 0] = 0.0
    v = torch.fft.ifftn(x * f).real
    return (v * (10.0 / v.std())).cpu().numpy()


# ---------------------------------------------------------------- prepare
class _State:
    """A context and what hangs on it, closed in order when the state goes."""

    def __init__(self, case):
        self.case = case
        self.ctx = abi.Context(0)
        self.dir = None
        self.sim = None

    def folder(self):
        self.dir = tempfile.TemporaryDirectory()
        return self.dir.name

    def __del__(self):
        if sys.is_finalizing():
            return
        if self.sim is not None:
            self.sim.close()
        self.ctx.close()


def prepare(case, seed):
    s, c = _State(case), case
    rng = np.random.default_rng(seed)
    kind = c["kind"]
    if kind == "forces":
        s.system, s.keep = _system(*_molecule(rng, c["atoms"], (0, 0), "buckled"), True, c["vdw"])
        s.ctx.set_systems([s.system])
        s.pos = _tip_points(c, rng)
    elif kind == "scan":
        s.system, s.keep = _system(*_molecule(rng, c["atoms"], _span(c), c["shape"]), c["coulomb"], "lj")
        s.desc = _scan_desc(c)
    elif kind == "batch":
        sizes = np.linspace(c["nmin"], c["nmax"], c["molecules"]).round().astype(int)
        made = [_system(*_molecule(rng, int(n), _span(c), "planar"), True, "lj") for n in rng.permutation(sizes)]
        s.keep = made
        s.ctx.set_systems([d for d, _ in made])
        s.desc = _scan_desc(c, c["precision"])
        s.records = torch.zeros(c["molecules"] * c["nx"] * c["ny"] * c["nz"], 11, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
    elif kind == "rigidgrid":
        s.system, s.keep = _system(*_molecule(rng, c["atoms"], _span(c), "planar"), True, "morse")
        s.desc = _scan_desc(c)
        s.grid = abi.GridDesc()
        h = [SCAN["dx"] / 2, SCAN["dy"] / 2, SCAN["dz"] / 2]
        border = [int(math.ceil(1.5 / v)) for v in h]
        low = SCAN["zhigh"] - (c["nz"] - 1) * SCAN["dz"] - s.system.tip_dummy_d
        for a in range(3):
            s.grid.n[a] = 2 * (c[("nx", "ny", "nz")[a]] - 1) + 2 * border[a] + 1
            s.grid.basis[4 * a] = h[a]
            s.grid.offset[a] = (low if a == 2 else 0.0) - border[a] * h[a]
        s.last = None
    elif kind == "slab":
        n, cell = c["atoms"], c["cell"]
        m = int(math.ceil(math.sqrt(n / 3)))
        lattice = np.stack(np.meshgrid(*(np.arange(k) for k in (m, m, 3)), indexing="ij"), -1).reshape(-1, 3)
        lattice = lattice[np.sort(rng.permutation(len(lattice))[:n])] + rng.uniform(-0.2, 0.2, (n, 3))
        pos = lattice * np.array([cell / m, cell / m, 1.5]) + np.array([0.0, 0.0, 0.5])
        types = list(rng.choice(["C", "N", "O", "H"], size=n, p=[0.5, 0.15, 0.10, 0.25]))
        shifts = np.array([[i * cell, j * cell, 0.0] for i in (-1, 0, 1) for j in (-1, 0, 1)])
        s.system, s.keep = _system(types, pos, np.zeros(n), False, "lj", shifts, [cell, cell, 20.0])
        ng = (c["n_grid"], c["n_grid"], 80)
        cube = _cube(dict(n0=ng[0], n1=ng[1], n2=ng[2]), rng)
        s.system.potential_grid = s.ctx.potential_grid(cube, np.diag([cell / ng[0], cell / ng[1], 0.25]),
                                                       np.zeros(3), ATOMS[TIP][3])
        # pixels spread over the whole cell, as the 256 x 256 image's are
        s.desc = _scan_desc(c, dx=cell / c["nx"], dy=cell / c["ny"], zhigh=14.4)
    elif kind == "gradient":
        w = workloads.make_c5(s.folder(), seed=int(rng.integers(1 << 30)), area="%g %g" % (c["area"], c["area"]),
                              zlow=c["zlow"])
        s.model = ScanModel(w.input_path, s.ctx)
        s.sim = s.model.sim
        s.target = torch.from_numpy(rng.normal(0.0, 0.3, int(np.prod(s.model.shape))))
    elif kind == "potential":
        s.cube = _cube(c, rng)
        s.basis = np.diag([0.25, 0.25, 0.25])
    elif kind == "flexible":
        w = workloads.make_fx_example(s.folder(), area="%g %g" % (c["ax"], c["ay"]), zlow=c["zlow"])
        xyz = os.path.join(s.dir.name, w.options["xyzfile"])
        head, *rows = [r.split() for r in open(xyz).read().splitlines()]
        with open(xyz, "w") as f:
            f.write(" ".join(head) + "\n\n")
            for r in rows:
                if r:
                    p = [float(v) + d for v, d in zip(r[1:4], rng.uniform(-0.005, 0.005, 3))]
                    f.write("%s %.5f %.5f %.5f %s\n" % (r[0], *p, " ".join(r[4:])))
        s.sim = abi.Simulation(w.input_path, s.ctx)
    else:
        w = workloads.make_fx(s.folder(), seed=int(rng.integers(1 << 30)))
        s.sim = abi.Simulation(w.input_path, s.ctx)
        fl = s.sim.flex_system()
        s.terms, s.fixed = fl["terms"], fl["fixed"]
        n, ns = fl["n_atoms"], c["states"]
        pos = np.repeat(fl["positions"][None], ns, 0)
        pos[:, 2:] += rng.normal(0.0, 0.01, (ns, n - 2, 3)) * (s.fixed[2:] != 1)[:, None]
        mid = fl["positions"][2:].mean(0)
        top = fl["positions"][2:, 2].max()
        pos[:, 0, :2] = mid[:2] + rng.uniform(-3, 3, (ns, 2))
        pos[:, 0, 2] = top + rng.uniform(6.5, 9.0, ns)
        pos[:, 1] = pos[:, 0] - np.array([0.0, 0.0, fl["tip_dummy_d"]])
        s.pos, s.vel = pos, np.zeros((ns, n, 3))
    return s


# ---------------------------------------------------------------- run
def run(s):
    c, ctx = s.case, s.ctx
    kind = c["kind"]
    if kind == "forces":
        return ctx.eval_tip_surface(0, s.pos)
    if kind in ("scan", "slab"):
        ctx.set_systems([s.system])
        ctx.scan(s.desc)
        out = _fields(ctx.records(0, c["nx"] * c["ny"] * c["nz"]))
        if c.get("deltaf"):
            out["deltaf"], out["z_low"] = ctx.delta_f(0, c["nx"], c["ny"], c["nz"], SCAN["zhigh"], SCAN["dz"])
        return out
    if kind == "batch":
        st = abi.ScanStats()
        ctx.check(abi.lib().mafm_scan_noalloc(ctx.h, ctypes.byref(s.desc), s.records.data_ptr(), len(s.records),
                                              ctypes.byref(st)))
        return {"records": s.records[:, :10], "steps_flags": s.records[:, 10:].view(torch.int32)}
    if kind == "rigidgrid":
        h = ctypes.c_int(-1)
        s.system.force_grid = -1
        ctx.check(abi.lib().mafm_grid_build(ctx.h, ctypes.byref(s.system), ctypes.byref(s.grid), ctypes.byref(h)))
        s.system.force_grid = h.value
        ctx.set_systems([s.system])
        if s.last is not None:
            ctx.grid_free(s.last)
        s.last = h.value
        ctx.scan(s.desc)
        return _fields(ctx.records(0, c["nx"] * c["ny"] * c["nz"]))
    if kind == "gradient":
        m = s.model
        leaves = [t.clone().requires_grad_(True) for t in (m.eps, m.sig, m.q, m.pos)]
        image = m.image(*leaves)
        ((image - s.target) ** 2).sum().backward()
        return {"image": image.detach(), "grads": [t.grad for t in leaves]}
    if kind == "potential":
        h = ctx.potential_grid(s.cube, s.basis, np.zeros(3), ATOMS[TIP][3])
        out = ctx.grid_download(h, s.cube.shape)
        ctx.grid_free(h)
        return out
    if kind == "flexible":
        s.sim.run("fast64")
        return _fields(s.sim.records())
    # the operator may work in the arrays it is given
    return list(ctx.system_minimise(s.terms, s.fixed, s.pos.copy(), s.vel.copy(), etol=0.01, ftol=0.01, dt=0.001, minterm=2))


# ---------------------------------------------------------------- work
def work(c):
    """Model of one pass: records written and tables read once; per FIRE
    iteration and evaluation ~30 FLOPs a site and ~100 for the tip, with the
    hundred iterations a height takes."""
    kind = c["kind"]
    if kind == "forces":
        return {"bytes": 56.0 * c["points"] + 64.0 * c["atoms"], "flops": 35.0 * c["atoms"] * c["points"]}
    if kind in ("scan", "batch", "slab", "rigidgrid", "gradient"):
        if kind == "gradient":
            n = (int(c["area"] / 0.1) + 1) ** 2 * (int((10.0 - c["zlow"]) / 0.1) + 1)
        else:
            n = c["nx"] * c["ny"] * c["nz"] * c.get("molecules", 1)
        sites = {"slab": 9 * c.get("atoms", 0), "batch": (c.get("nmin", 0) + c.get("nmax", 0)) / 2, "rigidgrid": 1,
                 "gradient": 150}.get(kind, c.get("atoms", 0))
        evals = {0: 1, 1: 2, 2: 4}[c.get("integrator", 1)]
        return {"bytes": 88.0 * n, "flops": 100.0 * n * (evals * (30.0 * sites + 50.0) + 52.0)}
    if kind == "potential":
        n = c["n0"] * c["n1"] * c["n2"]
        return {"bytes": 40.0 * n, "flops": 6 * 5.0 * n * math.log2(max(n, 2))}
    if kind == "flexible":
        n = (int(c["ax"] / 0.5) + 1) * (int(c["ay"] / 0.5) + 1) * (int((10.0 - c["zlow"]) / 0.1) + 1)
        return {"bytes": 88.0 * n, "flops": 150.0 * n * 2 * 40000.0}
    return {"bytes": 41 * 160.0 * c["states"], "flops": 100.0 * c["states"] * 2 * 20000.0}


# ---------------------------------------------------------------- exact
def exact(case, seed):
    c = case
    rng = np.random.default_rng(seed)
    if c["kind"] == "forces":
        if c["atoms"] * c["points"] > 3e7:
            return None
        types, pos, q = _molecule(rng, c["atoms"], (0, 0), "buckled")
        p, qq = _constants(types, q, True, c["vdw"])
        return _pairs(_tip_points(c, rng), pos, p, qq, c["vdw"])
    if c["kind"] == "scan" and c["nx"] * c["ny"] * c["atoms"] <= 10000 and c["integrator"] == 1:
        types, pos, q = _molecule(rng, c["atoms"], _span(c), c["shape"])
        p, qq = _constants(types, q, c["coulomb"], "lj")
        return dict(_fire_curves(c, pos, p, qq), **({"deltaf": None, "z_low": None} if c["deltaf"] else {}))
    if c["kind"] == "potential":
        return _potential(_cube(c, rng), 0.25, ATOMS[TIP][3], 0.5)
    return None


def _pairs(x, pos, p, qq, vdw):
    """Sum of the pair terms at points x: fx, fy, fz, e."""
    out = np.zeros((len(x), 4))
    for a in range(0, len(x), 4096):
        d = x[a:a + 4096, None, :] - pos[None]
        r = np.sqrt((d ** 2).sum(-1))
        if vdw == "lj":
            r6 = r ** 6
            e, f = p[:, 1] / r6 ** 2 - p[:, 0] / r6, (12 * p[:, 1] / r6 ** 2 - 6 * p[:, 0] / r6) / r ** 2
        else:
            w = np.exp(-p[:, 1] * (r - p[:, 2]))
            e, f = p[:, 0] * (w * w - 2 * w + 1), 2 * p[:, 0] * p[:, 1] * (w * w - w) / r
        e, f = e + qq / r, f + qq / r ** 3
        out[a:a + 4096, :3] = (f[..., None] * d).sum(1)
        out[a:a + 4096, 3] = e.sum(1)
    return out


def _fire_curves(c, pos, p, qq):
    """The scan in numpy: FIRE with the midpoint step, all columns at once,
    each column's state frozen once it has converged at a height."""
    S = SCAN
    es6, es12, _, sig = _mix(TIP, DUMMY)
    tip = np.array([[es6, es12, 0.0]])
    k = workloads.HARM[0]
    ij = np.stack(np.meshgrid(np.arange(c["nx"]), np.arange(c["ny"]), indexing="ij"), -1).reshape(-1, 2)
    n = len(ij)
    dummy = np.concatenate([ij * np.array([S["dx"], S["dy"]]), np.full((n, 1), S["zhigh"])], 1)
    t = dummy - np.array([0.0, 0.0, sig * 2 ** (1 / 6)])
    v, e = np.zeros((n, 3)), np.zeros(n)

    def total(x, live):
        fe = _pairs(x, pos, p, qq, "lj")
        for i in np.flatnonzero(live):
            fe[i] += _pairs(x[i:i + 1], dummy[i:i + 1], tip, np.zeros(1), "lj")[0]
        d = x - dummy
        fe[:, :2] -= 2 * k * d[:, :2]
        fe[:, 3] += k * (d[:, :2] ** 2).sum(1)
        return fe

    out = {f: np.zeros((n, c["nz"])) for f in ("x", "y", "z", "fx", "fy", "fz", "rx", "ry", "rz", "e")}
    for z in range(c["nz"]):
        dt, alpha, good = np.full((n, 1), S["dt"]), np.full((n, 1), 0.1), np.zeros((n, 1), int)
        live = np.ones(n, bool)
        for _ in range(1, S["maxsteps"]):
            f1 = total(t, live)[:, :3]
            fe = total(t + dt / 2 * v, live)
            t1, v1, f = t + dt * (v + dt / 2 * f1), v + dt * fe[:, :3], fe[:, :3]
            t, e_old, e = np.where(live[:, None], t1, t), e, np.where(live, fe[:, 3], e)
            fl = np.sqrt((f ** 2).sum(1))
            v = np.where(live[:, None], v1, v)
            live &= ~((np.abs(e - e_old) < S["etol"]) & (fl < S["ftol"]))
            if not live.any():
                break
            power = (v * f).sum(1, keepdims=True)
            mixed = (1 - alpha) * v + alpha * f / fl[:, None] * np.sqrt((v ** 2).sum(1, keepdims=True))
            m, up = live[:, None], power >= 0
            v = np.where(m, np.where(up, mixed, 0.0), v)
            fast = up & (good > 5)
            dt = np.where(up, np.where(fast, np.minimum(dt * 1.1, 10 * S["dt"]), dt), 0.5 * dt)
            alpha = np.where(up, np.where(fast, 0.99 * alpha, alpha), 0.1)
            good = np.where(up, good + 1, 0)
        fe = _pairs(t, pos, p, qq, "lj")
        out["x"][:, z], out["y"][:, z], out["z"][:, z] = dummy.T
        out["fx"][:, z], out["fy"][:, z], out["fz"][:, z], out["e"][:, z] = fe.T
        out["rx"][:, z], out["ry"][:, z], out["rz"][:, z] = (t - dummy).T
        dummy, t = dummy - np.array([0.0, 0.0, S["dz"]]), t - np.array([0.0, 0.0, S["dz"]])
    return dict({f: a.ravel() for f, a in out.items()}, n_steps=None, flags=None)


def _potential(cube, h, charge, width):
    """Energy and force of a Gaussian charge in the potential: convolution and
    spectral gradient, the Gaussian cut where it falls below 1e-10."""
    n = cube.shape
    cut = next((i for i in range(min(n) - 1) if math.exp(-0.5 * (i * h) ** 2 / width ** 2) < 1e-10), min(n))
    i, z = np.arange(-cut, cut + 1), np.arange(-cut, cut)
    g = np.exp(-0.5 * h * h / width ** 2 * (i[:, None, None] ** 2 + i[None, :, None] ** 2 + z[None, None, :] ** 2))
    rho = np.zeros(n)
    np.add.at(rho, (i[:, None, None] % n[0], i[None, :, None] % n[1], z[None, None, :] % n[2]), g)
    rho *= charge / (width * math.sqrt(2 * math.pi)) ** 3
    ek = np.fft.fftn(cube) * h ** 3 * np.fft.fftn(rho)
    out = np.zeros(n + (4,))
    out[..., 3] = np.fft.ifftn(ek).real
    for a in range(3):
        k = np.arange(n[a], dtype=float)
        k[k >= n[a] // 2] -= n[a]
        k = (k / (n[a] * h)).reshape([-1 if b == a else 1 for b in range(3)])
        out[..., a] = np.fft.ifftn(-2j * math.pi * k * ek).real
    return out.reshape(-1, 4)
