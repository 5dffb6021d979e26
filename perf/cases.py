"""The work that programs have this library do, as cases to be timed: whole time steps in
every solver and precision, the pressure solve on its own, the explicit stages, and the drag
adjoint, from the 128 x 64 x 4 grid to 1024 x 512 x 128.

A case is a dict of plain values.  `kind` says what one pass does:
  steps    a short run: the seeded initial field, `steps` time steps, the fields read back
  solve    one pressure solve of a right-hand side the program hands over, x read back
  stages   the explicit stages of `steps` steps called one by one, the fields read back
  adjoint  the mean drag over `steps` steps and its gradients, checkpoints every `every`
`iters` is the number of pressure iterations (or red-black sweeps) a step is expected to
take; it enters `work` only.
"""
import math

import numpy as np

import cfd_nssolver_forhpc_flowpassingcylinder_amd as pkg
from cfd_nssolver_forhpc_flowpassingcylinder_amd.api import (GRID_SML, GRID_UNIFORM,
                                                             PRECISION_FP64, PRECISION_FP64_MG,
                                                             PRECISION_MIXED, SOLVER_BICGSTAB,
                                                             SOLVER_RBSOR)

PRECISIONS = {"fp64": PRECISION_FP64, "mixed": PRECISION_MIXED, "fp64_mg": PRECISION_FP64_MG}

# faces x- x+ y- y+ z- z+, components u v w: inflow, outflow and slip walls
SLIP_NUM = [[0, 0, 0], [1, 1, 1], [1, 0, 1], [1, 0, 1], [1, 1, 1], [1, 1, 1]]
SLIP_DIR = [[1, 0, 0]] + [[0, 0, 0]] * 5

_BASE = dict(lx=20.0, ly=10.0, lz=0.5, sml=False, periodic=True, precision="fp64",
             rbsor=False, jacobi=False, cs=0.0, re=200.0, dt=0.001, tol=1e-10, maxit=5000,
             steps=1, every=1, iters=0)


def _case(name=None, **kw):
    c = dict(_BASE, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the CPU-runnable configuration: Jacobi-scaled rows, a few hundred iterations a step,
        # every launch small
        _case("fp64_128x64x4", kind="steps", nx=128, ny=64, nz=4, re=100.0, dt=0.002, tol=1e-8,
              jacobi=True, steps=4, iters=340),
        # the reference's own stretched grid with walls at its default tolerance
        _case("fp64_sml_112x104x4", kind="steps", nx=112, ny=104, nz=4, lx=17.0, ly=12.0,
              lz=3.0, sml=True, periodic=False, re=100.0, dt=0.002, tol=1e-3, maxit=1000,
              steps=4, iters=200),
        # a pressure solve called on its own (what the drop-in's solver entry does), at the
        # size of the adjoint configuration
        _case("solve_fp64_256x128x32", kind="solve", nx=256, ny=128, nz=32, re=100.0,
              dt=0.002, iters=1500),
        # the headline configuration in plain FP64, the solve bounded by its iteration limit
        _case("fp64_512x256x64", kind="steps", nx=512, ny=256, nz=64, maxit=1500, steps=2,
              iters=1500),
        # sizes off every power of two, walled z, odd nz
        _case("fp64_odd_197x93x31", kind="steps", nx=197, ny=93, nz=31, periodic=False,
              re=150.0, tol=1e-6, maxit=600, steps=2, iters=600),
        # red-black SOR at its sweep limit
        _case("rbsor_512x256x64", kind="steps", nx=512, ny=256, nz=64, rbsor=True, maxit=1000,
              steps=2, iters=1000),
        # the production mode: mixed precision from the seeded field
        _case("mixed_512x256x64", kind="steps", nx=512, ny=256, nz=64, precision="mixed",
              steps=10, iters=5),
        # the same algorithm in FP64
        _case("fp64mg_256x128x32", kind="steps", nx=256, ny=128, nz=32, re=100.0, dt=0.002,
              precision="fp64_mg", steps=20, iters=5),
        # small multigrid levels throughout, z walled, nz even but no multiple of four
        _case("mixed_96x48x6", kind="steps", nx=96, ny=48, nz=6, lz=1.25, precision="mixed",
              periodic=False, steps=20, iters=6),
        # the large configuration
        _case("mixed_1024x512x128", kind="steps", nx=1024, ny=512, nz=128, re=3900.0,
              dt=0.0005, precision="mixed", steps=4, iters=6),
        # the explicit stages of a large-eddy run, called one by one
        _case("stages_les_384x192x48", kind="stages", nx=384, ny=192, nz=48, re=3900.0,
              dt=0.0005, cs=0.18, steps=20),
        # drag gradients, checkpoint and recompute, multigrid pressure solves
        _case("adjoint_256x128x32", kind="adjoint", nx=256, ny=128, nz=32, re=100.0, dt=0.002,
              precision="fp64_mg", steps=10, every=5, iters=5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _coarsens(n, h):
    """Whether halving the directions whose spacing is within twice the smallest takes the
    grid to at most 512 cells, as the multigrid modes ask."""
    n, h = list(n), list(h)
    while n[0] * n[1] * n[2] > 512:
        m = 2.0 * min(h)
        can = [h[q] <= m and n[q] % 2 == 0 and n[q] >= (2 if q == 2 else 4) for q in range(3)]
        if not any(can):
            return False
        for q in range(3):
            if can[q]:
                n[q], h[q] = n[q] // 2, 2.0 * h[q]
    return True


def draw(rng):
    what = rng.choice(["fp64", "fp64", "solve", "rbsor", "mixed", "fp64_mg", "mixed", "stages",
                       "adjoint"])
    re, dt = rng.choice([100.0, 150.0, 200.0]), rng.choice([0.0005, 0.001])
    if what in ("mixed", "fp64_mg", "adjoint"):
        # a small box doubled a few times, until its halvings reach the coarsest level
        while True:
            k = rng.randint(2, 5 if what != "adjoint" else 3)
            nx = rng.choice([10, 12, 14, 16]) << k
            ny = rng.choice([4, 6, 7, 8]) << k
            nz = rng.choice([4, 6, 8, 12, 16, 24, 32] if rng.random() < 0.8 else [5, 7])
            # z cells as wide as x cells for odd nz, else also flatter ones
            lz = nz * 20.0 / nx / (1 if nz % 2 else rng.choice([1, 2, 4]))
            if _coarsens((nx, ny, nz), (20.0 / nx, 20.0 / nx, lz / nz)):
                break
        n = nx * ny * nz
        steps = max(2, min(12, 4_000_000 // n))
        return _case(kind="adjoint" if what == "adjoint" else "steps", nx=nx, ny=ny, nz=nz,
                     ly=20.0 * ny / nx, lz=lz, periodic=what == "adjoint" or rng.random() < 0.7,
                     precision=what if what != "adjoint" else rng.choice(["mixed", "fp64_mg"]),
                     re=re, dt=dt, steps=steps, every=rng.randint(1, steps), iters=6)
    nx, ny = _log(rng, 40, 420), _log(rng, 24, 210)
    nz = _log(rng, 4, 72)
    n = nx * ny * nz
    if what == "stages":
        return _case(kind="stages", nx=nx, ny=ny, nz=nz, cs=rng.choice([0.0, 0.1, 0.18]), re=re,
                     dt=dt, periodic=rng.random() < 0.6, steps=rng.randint(4, 16))
    if what == "solve":  # small enough to be solved to its tolerance
        nx, ny, nz = _log(rng, 24, 200), _log(rng, 16, 100), _log(rng, 4, 16)
        return _case(kind="solve", nx=nx, ny=ny, nz=nz, jacobi=rng.random() < 0.3,
                     periodic=rng.random() < 0.6, iters=700)
    its = max(20, min(400, 600_000_000 // n))
    if what == "rbsor":
        return _case(kind="steps", nx=nx, ny=ny, nz=nz + nz % 2, rbsor=True, re=re, dt=dt,
                     periodic=rng.random() < 0.6, maxit=its, steps=2, iters=its)
    return _case(kind="steps", nx=nx, ny=ny, nz=nz, re=re, dt=dt,
                 jacobi=rng.random() < 0.3, periodic=rng.random() < 0.6, maxit=its, steps=2,
                 iters=its)


def _solver(c):
    per = 1 if c["periodic"] else 0
    cfg = pkg.default_config(
        nx=c["nx"], ny=c["ny"], nz=c["nz"], lx=c["lx"], ly=c["ly"], lz=c["lz"],
        grid_kind=GRID_SML if c["sml"] else GRID_UNIFORM, re=c["re"], dt=c["dt"], tol=c["tol"],
        maxit=c["maxit"], solver=SOLVER_RBSOR if c["rbsor"] else SOLVER_BICGSTAB,
        precond=1 if c["jacobi"] else 0, sor_omega=1.8, z_periodic=per,
        precision=PRECISIONS[c["precision"]], smagorinsky_cs=c["cs"], skip_first_pressure=1)
    if not c["sml"]:  # the stretched grid keeps the reference's own boundary table
        for f in range(6):
            for q in range(3):
                cfg.bc_num[f][q] = SLIP_NUM[f][q]
                cfg.bc_dir[f][q] = SLIP_DIR[f][q]
        if per:
            cfg.outflow_convective, cfg.convective_speed, cfg.flux_correction = 1, 1.0, 1
        else:  # closed z walls, so that the outlet's flux can be corrected
            for f in (4, 5):
                cfg.bc_num[f][2] = 0.0
            cfg.flux_correction = 1
    return pkg.FlowSolver(cfg)


def _rhs(c, seed):
    """A right-hand side as a step leaves it: smooth, with a source at the cylinder and a
    little noise, mean-free."""
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    rng = np.random.default_rng(seed)
    x = (np.arange(nx) + 0.5) * c["lx"] / nx
    y = (np.arange(ny) + 0.5) * c["ly"] / ny
    z = (np.arange(nz) + 0.5) / nz
    a, b = rng.uniform(4.5, 5.5, 2)
    r2 = ((x - a) ** 2)[:, None] + ((y - b * c["ly"] / 10.0) ** 2)[None, :]
    f = (np.exp(-4.0 * r2) * (x - a)[:, None])[:, :, None] * (1 + 0.1 * np.cos(2 * np.pi * z))
    f = f + 1e-3 * rng.standard_normal((nx, ny, nz))
    return np.ascontiguousarray(f - f.mean()).reshape(-1)


def prepare(case, seed):
    s = _solver(case)
    cy = case["ly"] / 2.0
    if case["kind"] == "adjoint":
        rng = np.random.default_rng(seed)
        s.set_inflow(1.0 + 0.01 * rng.standard_normal(s.ny))
        s.set_eta_smoothed(5.0, cy, 0.5, 0.75 * case["lx"] / case["nx"])
        s.init_flow(1.0, 1e-3, seed)
    elif case["kind"] == "solve":
        s.init_flow(1.0, 1e-3, seed)
        return dict(case=case, s=s, rhs=_rhs(case, seed), x0=np.zeros(s.N))
    else:
        s.set_eta_cylinder_z(6.5 if case["sml"] else 5.0, cy, 0.5, 100)
    return dict(case=case, s=s, seed=seed)


def run(state):
    c, s = state["case"], state["s"]
    if c["kind"] == "solve":
        s.set_rhs(state["rhs"])
        s.set_xresult(state["x0"])
        iters, _ = s.solve_bicgstab()
        return dict(iters=iters, x=s.xresult())
    if c["kind"] == "adjoint":
        J, gi, gm, info = s.adjoint_drag(c["steps"], c["every"])
        return dict(J=J, inflow=gi, mask=gm, iters=[info["forward_iters"], info["adjoint_iters"]])
    s.init_flow(1.0, 1e-3, state["seed"])
    if c["kind"] == "stages":
        for _ in range(c["steps"]):
            if c["cs"] > 0.0:
                s.smagorinsky()
            s.convdiff()
            s.pressure_rhs()
            s.project_ib()
            s.swap_t0_t3()
            s.bc_main()
            s.bc_copy()
        return dict(cfl=s.cfl(), drag=list(s.cd_cl()), u=list(s.download_velocity(0)),
                    rhs=s.rhs(), f=s.force())
    info = s.step(c["steps"])
    return dict(iters=info["iters"], cd=info["cd"], cl=info["cl"], cfl=info["cfl"],
                u=list(s.download_velocity(0)), p=s.pressure())


def exact(case, seed):
    """The pressure solve's solution by the eigenvectors of the uniform operator's three
    one-dimensional chains, mean-free as the iteration keeps it; no value for the other
    kinds, which integrate a nonlinear flow."""
    if case["kind"] != "solve" or case["jacobi"]:
        return None
    f = _rhs(case, seed).reshape(case["nx"], case["ny"], case["nz"])
    qs, lams = [], []
    for n, ln, periodic in ((case["nx"], case["lx"], False), (case["ny"], case["ly"], False),
                            (case["nz"], case["lz"], case["periodic"])):
        a = np.zeros((n, n))
        for i in range(n):
            for m in (i - 1, i + 1):
                if 0 <= m < n or periodic:
                    a[i, i] += 1.0
                    a[i, m % n] -= 1.0
        lam, q = np.linalg.eigh(a * (n / ln) ** 2)
        qs.append(q)
        lams.append(lam)
    c = np.einsum("ia,ijk->ajk", qs[0], f, optimize=True)
    c = np.einsum("jb,ajk->abk", qs[1], c, optimize=True)
    c = np.einsum("kc,abk->abc", qs[2], c, optimize=True)
    lam = lams[0][:, None, None] + lams[1][None, :, None] + lams[2]
    lam[0, 0, 0] = 1.0
    c = c / lam
    c[0, 0, 0] = 0.0
    c = np.einsum("ia,abc->ibc", qs[0], c, optimize=True)
    c = np.einsum("jb,ibc->ijc", qs[1], c, optimize=True)
    c = np.einsum("kc,ijc->ijk", qs[2], c, optimize=True)
    return dict(iters=None, x=c.reshape(-1))


def work(case):
    n, g = case["nx"] * case["ny"] * case["nz"], 1
    for q in ("nx", "ny", "nz"):
        g *= case[q] + 4
    # FP64 values per cell and step that the explicit part cannot do without: the velocity
    # read and written, u* written and read, the pressure and forcing written, the mask read
    step = (6 + 6 + 4 + 1) * 8.0
    if case["rbsor"]:
        it, flop = 24.0, 16.0  # per sweep: p read and written, the right-hand side read
    elif case["precision"] == "fp64":
        it, flop = 56.0, 46.0  # per iteration: x, r and q read and written, r0 read
    else:
        t = 4.0 if case["precision"] == "mixed" else 8.0
        # two V(2,2) cycles: right-hand side and correction of every level (at most 2 n
        # cells in all) each read and written once on the way down and up, and the vectors
        it, flop = t * (2 * 2 * 6 + 12) + 16.0, 2 * 2 * 5 * 14.0
    out = 8.0 * 4 * g
    if case["kind"] == "solve":
        return dict(bytes=case["iters"] * it * n + 32.0 * n, flops=case["iters"] * flop * n)
    if case["kind"] == "stages":
        return dict(bytes=case["steps"] * step * n + 8.0 * 7 * g, flops=case["steps"] * 700.0 * n)
    per = step + case["iters"] * it
    steps = case["steps"] * (2 if case["kind"] == "adjoint" else 1)
    return dict(bytes=steps * per * n + out, flops=steps * (700.0 + case["iters"] * flop) * n)
