"""The work that is timed when this library is made faster.

Each case is one pass through the public entry points (the Python mirror of
the reference's API, or the C ABI it binds), as a solver program calls them:

  kind "simple"     SIMPLE iterations of a laminar case (cavity or backward-
                    facing step), FP64 or mixed precision
  kind "komega"     SIMPLE iterations of the k-omega flat plate
  kind "batch"      one iteration of many independent cases advanced together
  kind "transport"  scalar transport on a Delaunay triangulation: assembly,
                    boundary conditions, relaxation, DILU update, BiCGSTAB
  kind "pressure"   the pressure corrector's equation on a quad grid: assembly
                    with a face coefficient and a source, boundary conditions,
                    preconditioner update, Krylov solve
  kind "assemble"   the momentum-like equation's assembly alone
  kind "gradient"   a cell gradient with its face interpolation

The solves of "transport" and "pressure" run a fixed number of iterations
(their tolerance is out of reach), so that a pass is the same work for all
inputs of a case.
"""
import ctypes as C
import functools
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "xcalibre_tw.jl_amd"))

import fvmhip as F  # noqa: E402
from fvmhip import _lib as L  # noqa: E402

PRECISION = {"fp64": L.FP64, "mixed": L.MIXED}
SOLVER = {"cg": F.CgSolver, "bicgstab": F.BicgstabSolver, "gmres": F.GmresSolver}
PRECOND = {"dilu": F.DILU, "ilu0": F.ILU0, "jacobi": F.Jacobi, "ldl": F.LDL}
GRADIENT = {"orthogonal": F.Orthogonal, "midpoint": F.Midpoint}
RELAX = 0.8
DIVERGENCE = {"linear": F.Linear, "upwind": F.Upwind}


def listed():
    return [
        # the smallest whole run: the 40 x 40 lid-driven cavity of the reference's first tutorial
        {"name": "cavity 40 fp64", "kind": "simple", "mesh": "cavity", "nx": 40, "ny": 40, "precision": "fp64",
         "iterations": 150},
        # the benchmark of this repository: SIMPLE on the 2000 x 500 backward-facing step
        {"name": "step 2000x500 fp64", "kind": "simple", "mesh": "step", "nx": 2000, "ny": 500, "precision": "fp64",
         "iterations": 2},
        # turbulent flow with wall functions, five solves per iteration, mixed-precision U and p
        {"name": "plate 1000x500 mixed", "kind": "komega", "nx": 1000, "ny": 500, "precision": "mixed",
         "iterations": 2},
        # a parameter study: many small cases of uneven size in one launch per phase
        {"name": "batch 24", "kind": "batch", "count": 24, "lo": 32, "hi": 256, "pick": 5, "precision": "fp64"},
        # scalar transport on unstructured meshes, ordinary and large, both precisions
        {"name": "transport 30k fp64", "kind": "transport", "points": 30011, "precision": "fp64", "itmax": 15},
        {"name": "transport 250k mixed", "kind": "transport", "points": 250007, "precision": "mixed", "itmax": 6},
        # the pressure equation with each preconditioner of the user API: the reference's step case
        # runs GMRES + LDL, its defaults CG + DILU; an odd ragged grid, a mid-size and a large one
        {"name": "pressure gmres ldl 400x100", "kind": "pressure", "nx": 400, "ny": 100, "solver": "gmres",
         "precond": "ldl", "itmax": 10, "precision": "fp64"},
        {"name": "pressure cg dilu 317x203", "kind": "pressure", "nx": 317, "ny": 203, "solver": "cg",
         "precond": "dilu", "itmax": 40, "precision": "fp64"},
        {"name": "pressure bicgstab ilu0 250x125", "kind": "pressure", "nx": 250, "ny": 125, "solver": "bicgstab",
         "precond": "ilu0", "itmax": 10, "precision": "fp64"},
        {"name": "pressure cg jacobi 1500x1000", "kind": "pressure", "nx": 1500, "ny": 1000, "solver": "cg",
         "precond": "jacobi", "itmax": 50, "precision": "fp64"},
        # the two largest operators of an iteration besides the solves
        {"name": "assemble 2000x1000", "kind": "assemble", "mesh": "quads", "nx": 2000, "ny": 1000,
         "divergence": "upwind"},
        {"name": "gradient 250k points", "kind": "gradient", "mesh": "triangles", "points": 250007,
         "scheme": "orthogonal"},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["simple", "komega", "batch", "transport", "pressure", "pressure", "pressure", "assemble",
                       "gradient"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "simple":
        if rng.random() < 0.5:
            n = _log_int(rng, 20, 300)
            return {"kind": kind, "mesh": "cavity", "nx": n, "ny": n, "precision": precision, "iterations": 8}
        return {"kind": kind, "mesh": "step", "nx": _log_int(rng, 60, 2000), "ny": _log_int(rng, 20, 500),
                "precision": precision, "iterations": 2}
    if kind == "komega":
        return {"kind": kind, "nx": _log_int(rng, 60, 1000), "ny": _log_int(rng, 30, 500), "precision": precision,
                "iterations": 2}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(3, 24), "lo": 32, "hi": 256, "pick": rng.randint(0, 999),
                "precision": precision}
    if kind == "transport":
        return {"kind": kind, "points": _log_int(rng, 500, 250000), "precision": precision,
                "itmax": rng.randint(3, 6) if precision == "mixed" else rng.randint(5, 15)}
    if kind == "pressure":
        pre = rng.choice(["dilu", "dilu", "ilu0", "jacobi", "ldl"])
        hi = {"dilu": (1500, 1000), "jacobi": (1500, 1000), "ilu0": (300, 150), "ldl": (400, 100)}[pre]
        mixed = precision == "mixed" and pre != "ldl"
        solver = rng.choice(["cg", "bicgstab", "gmres"])
        # (BiCGSTAB amplifies rounding from iteration to iteration: few of them, as in its use)
        itmax = 10 if pre in ("ldl", "ilu0") else rng.randint(10, 40) if solver != "bicgstab" else rng.randint(5, 15)
        if mixed and solver == "bicgstab":
            itmax = rng.randint(3, 6)
        return {"kind": kind, "nx": _log_int(rng, 30, hi[0]), "ny": _log_int(rng, 17, hi[1]), "solver": solver,
                "precond": pre, "itmax": itmax, "precision": "mixed" if mixed else "fp64"}
    if kind == "assemble":
        if rng.random() < 0.5:
            return {"kind": kind, "mesh": "quads", "nx": _log_int(rng, 40, 2000), "ny": _log_int(rng, 40, 1000),
                    "divergence": rng.choice(["upwind", "linear"])}
        return {"kind": kind, "mesh": "triangles", "points": _log_int(rng, 500, 250000),
                "divergence": rng.choice(["upwind", "linear"])}
    scheme = rng.choice(["orthogonal", "midpoint"])
    if rng.random() < 0.5:
        return {"kind": kind, "mesh": "quads", "nx": _log_int(rng, 40, 2000), "ny": _log_int(rng, 40, 1000),
                "scheme": scheme}
    return {"kind": kind, "mesh": "triangles", "points": _log_int(rng, 500, 250000), "scheme": scheme}


# ---------------------------------------------------------------------------
# Meshes: a program makes its mesh once and runs many inputs on it
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=16)
def _mesh(key):
    what, *size = key
    if what == "cavity":
        return F.cavity(size[0])
    if what == "step":
        return F.backward_facing_step(nx=size[0], ny=size[1], grading=1.02 if size[1] >= 100 else 1.0)
    if what == "plate":
        # first cell and growth that fit the height whatever the cell count
        return F.flat_plate(nx=size[0], ny=size[1], first=4.0e-5, ratio=1.05)
    if what == "quads":
        return F.channel(size[0], size[1], lx=2.0, ly=1.0, grading=1.002)
    return F.delaunay_unit_square(size[0], seed=0)


@functools.lru_cache(maxsize=1)
def _batch_models(count, lo, hi, pick):
    rng = np.random.default_rng(pick)
    sides = np.rint(np.exp(rng.uniform(np.log(lo), np.log(hi), count))).astype(int)
    return [F.cavity(int(n)) if k % 2 == 0 else F.channel(int(n), int(n)) for k, n in enumerate(sides)]


def _mesh_of(case):
    if case["kind"] == "simple":
        return _mesh((case["mesh"],) + ((case["nx"],) if case["mesh"] == "cavity" else (case["nx"], case["ny"])))
    if case["kind"] == "komega":
        return _mesh(("plate", case["nx"], case["ny"]))
    if case["kind"] == "pressure" or case.get("mesh") == "quads":
        return _mesh(("quads", case["nx"], case["ny"]))
    return _mesh(("triangles", case["points"]))


def _cells(case):
    k = case["kind"]
    if k == "batch":
        rng = np.random.default_rng(case["pick"])
        s = np.rint(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), case["count"])))
        return int((s * s).sum())
    if "points" in case:
        return 2 * case["points"]
    return case["nx"] * case["ny"]


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _smooth(xy, rng, modes=4, amplitude=1.0):
    """A smooth random field: a few Fourier modes."""
    out = np.zeros(xy.shape[0])
    for _ in range(modes):
        kx, ky = rng.integers(1, 5, 2)
        px, py, a = rng.uniform(0, 2 * np.pi, 2).tolist() + [rng.uniform(-1, 1)]
        out += a * np.sin(kx * xy[:, 0] + px) * np.cos(ky * xy[:, 1] + py)
    return amplitude * out


def _solenoidal_flux(mesh, rng):
    """Face fluxes of a smooth divergence-free velocity (a stream function's curl)."""
    x, y = mesh.face_centre[:, 0], mesh.face_centre[:, 1]
    u, v = np.zeros(x.size), np.zeros(x.size)
    for _ in range(3):
        k, m = rng.integers(1, 4, 2)
        a, p, q = rng.uniform(0.3, 1.0), *rng.uniform(0, 2 * np.pi, 2)
        u += a * m * np.sin(k * np.pi * x + p) * np.cos(m * np.pi * y + q)
        v -= a * k * np.cos(k * np.pi * x + p) * np.sin(m * np.pi * y + q)
    return mesh.face_area * (u * mesh.face_normal[:, 0] + v * mesh.face_normal[:, 1])


def _config(case, turbulent=False, iterations=1 << 20):
    precision = PRECISION[case["precision"]]
    scheme = F.set_schemes(divergence=F.Upwind)
    kw = dict(convergence=1e-7, itmax=100)
    solvers = dict(U=F.set_solver(None, solver=F.BicgstabSolver, preconditioner=F.DILU(), relax=0.7,
                                  precision=precision, **kw),
                   p=F.set_solver(None, solver=F.CgSolver, preconditioner=F.DILU(), relax=0.3, precision=precision,
                                  **kw))
    names = ["U", "p"]
    if turbulent:
        names += ["k", "omega"]
        for q in ("k", "omega"):
            solvers[q] = F.set_solver(None, solver=F.GmresSolver, preconditioner=F.DILU(), relax=0.7, **kw)
    return F.Configuration(schemes={q: scheme for q in names}, solvers=solvers,
                           runtime=F.set_runtime(iterations=iterations, write_interval=-1, time_step=1.0))


def _cavity(mesh, lid, nu):
    model = F.RANS(F.Laminar, mesh=mesh, viscosity=F.ConstantScalar(nu))
    z = [0.0, 0.0, 0.0]
    F.assign(model, "U", F.Dirichlet("inlet", z), F.Dirichlet("outlet", z), F.Dirichlet("bottom", z),
             F.Dirichlet("top", [lid, 0.0, 0.0]))
    F.assign(model, "p", *[F.Neumann(b, 0.0) for b in ("inlet", "outlet", "bottom", "top")])
    return model


def _channel(mesh, speed, nu, inlet=("inlet",), walls=("bottom", "top")):
    model = F.RANS(F.Laminar, mesh=mesh, viscosity=F.ConstantScalar(nu))
    z = [0.0, 0.0, 0.0]
    F.assign(model, "U", *[F.Dirichlet(b, [speed, 0.0, 0.0]) for b in inlet], F.Neumann("outlet", 0.0),
             *[F.Dirichlet(b, z) for b in walls])
    F.assign(model, "p", *[F.Neumann(b, 0.0) for b in inlet], F.Dirichlet("outlet", 0.0),
             *[F.Neumann(b, 0.0) for b in walls])
    F.initialise(model.U, [speed, 0.0, 0.0])
    return model


def _perturb(model, rng, amplitude):
    """Initial velocity with a smooth disturbance."""
    c = model.mesh.cell_centre
    xy = (c[:, :2] - c[:, :2].min(0)) / (np.ptp(c[:, :2], axis=0) + 1e-30) * np.pi
    model.U.x.values += _smooth(xy, rng, amplitude=amplitude)
    model.U.y.values += _smooth(xy, rng, amplitude=amplitude)


def _plate(mesh, speed, nu=1.5e-5):
    k_in = 1.5 * (0.01 * speed) ** 2
    w_in = k_in / (10.0 * nu)
    model = F.RANS(F.KOmega, mesh=mesh, viscosity=F.ConstantScalar(nu))
    z = [0.0, 0.0, 0.0]
    F.assign(model, "U", F.Dirichlet("inlet", [speed, 0.0, 0.0]), F.Neumann("outlet", 0.0), F.Dirichlet("wall", z),
             F.Neumann("top", 0.0))
    F.assign(model, "p", F.Neumann("inlet", 0.0), F.Dirichlet("outlet", 0.0), F.Neumann("wall", 0.0),
             F.Neumann("top", 0.0))
    for name, value, wall in (("k", k_in, F.KWallFunction), ("omega", w_in, F.OmegaWallFunction),
                              ("nut", k_in / w_in, F.NutWallFunction)):
        F.assign(model, name, F.Dirichlet("inlet", value), F.Neumann("outlet", 0.0), wall("wall"),
                 F.Neumann("top", 0.0))
        F.initialise(model.turbulence[name], value)
    F.initialise(model.U, [speed, 0.0, 0.0])
    return model


class _Owned:
    """Device memory of the library as torch sees it (no copy)."""

    def __init__(self, ptr, n):
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": "<f8", "data": (int(ptr), False), "version": 2}


class _Handle:
    """An fvh_eqn and what it needs alive; destroyed with its last user."""

    def __init__(self, mesh):
        self.mesh, self.h = mesh, C.c_void_p()
        L.check(L.lib().fvh_eqn_create(mesh.device().h, C.byref(self.h)), "fvh_eqn_create")

    def __del__(self):
        try:
            L.lib().fvh_eqn_destroy(self.h)
        except Exception:
            pass


def _tensor(handle, ptr, n):
    """The equation's array as a tensor, which keeps the equation alive."""
    t = torch.as_tensor(_Owned(ptr, n), device="cuda")
    if t.data_ptr() != ptr:
        raise RuntimeError("torch copied the library's array")
    t.owner = handle
    return t


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a, np.float64)).cuda()


def _p(t):
    return C.c_void_p(t.data_ptr())


def _copy(dst, src):
    L.check(L.lib().fvh_memcpy(_p(dst), _p(src), 8 * src.numel()), "fvh_memcpy")


class _Equation:
    """One equation on the device, driven through the C ABI call by call:
    sum of terms (operator, scheme, sign, face flux) == source."""

    def __init__(self, mesh, terms, source, bcs, phi):
        self.mesh, self.phi, self.keep = mesh, phi, (terms, source)
        nz, b = C.c_void_p(), C.c_void_p()
        self.handle = _Handle(mesh)
        self.h = self.handle.h
        L.check(L.lib().fvh_eqn_arrays(self.h, C.byref(nz), C.byref(b)))
        self.terms = (L.Term * len(terms))()
        for t, (op, scheme, sign, flux) in zip(self.terms, terms):
            t.op, t.scheme, t.sign, t.flux, t.phi = op, scheme, sign, flux.data_ptr(), phi.data_ptr()
        self.nterms = len(terms)
        self.src = (L.Source * 1)()
        self.nsrc = 0 if source is None else 1
        if source is not None:
            self.src[0].sign, self.src[0].field = 1, source.data_ptr()
        self.bcs = (L.BC * max(1, len(bcs)))()
        for t, bc in zip(self.bcs, bcs):
            t.kind, t.patch = bc.kind, mesh.boundary_index(bc.ID)
            for j in range(3):
                t.value[j] = float(bc.value)
        self.nbc = len(bcs)
        nnz = mesh.device().pattern()[1].size
        self.nz, self.b = _tensor(self.handle, nz.value, nnz), _tensor(self.handle, b.value, mesh.ncells)

    def discretise(self):
        L.check(L.lib().fvh_discretise(self.h, self.terms, self.nterms, self.src, self.nsrc, None, 1.0),
                "fvh_discretise")
        L.check(L.lib().fvh_apply_bcs(self.h, self.terms, self.nterms, self.bcs, self.nbc, 0), "fvh_apply_bcs")

    def precond(self, kind):
        L.check(L.lib().fvh_precond_set(self.h, kind.kind, None), "fvh_precond_set")

    def update(self):
        L.check(L.lib().fvh_precond_update(self.h), "fvh_precond_update")

    def solve(self, cfg):
        st = L.Stats()
        L.check(L.lib().fvh_solve(self.h, C.byref(cfg), _p(self.phi), C.byref(st)), "fvh_solve")
        return st


def _solver_cfg(case, solver, pre):
    return L.SolverCfg(solver=SOLVER[solver], precond=PRECOND[pre].kind, itmax=case["itmax"],
                       precision=PRECISION[case["precision"]], convergence=0.0, relax=1.0, atol=0.0,
                       rtol=1e-5 if case["precision"] == "mixed" else 1e-14)


def _host_inputs(case, mesh, seed):
    """The seeded arrays of the kinds that drive one equation (host)."""
    rng = np.random.default_rng([seed, 7])
    xy = np.pi * mesh.cell_centre[:, :2]
    fxy = np.pi * mesh.face_centre[:, :2]
    kind = case["kind"]
    if kind == "pressure":  # 1/a_P on the faces, the divergence of the predicted velocity as source
        return dict(gamma=np.exp(_smooth(fxy, rng, amplitude=0.4)), x0=_smooth(xy, rng, amplitude=0.1),
                    source=_smooth(xy, rng) + 0.05 * rng.standard_normal(mesh.ncells))
    if kind == "gradient":
        return dict(phi=_smooth(xy, rng) + 0.01 * rng.standard_normal(mesh.ncells), wall=float(rng.uniform(0.5, 1.5)))
    return dict(mdot=_solenoidal_flux(mesh, rng), gamma=1e-3 * np.exp(_smooth(fxy, rng, amplitude=0.3)),
                x0=_smooth(xy, rng, amplitude=0.1), source=_smooth(xy, rng), wall=float(rng.uniform(0.5, 1.5)))


def _bcs(case, mesh, h):
    kind = case["kind"]
    quads = "inlet" in mesh.boundary_names
    if kind == "pressure":
        return [F.Neumann("inlet", 0.0), F.Dirichlet("outlet", 0.0), F.Neumann("bottom", 0.0), F.Neumann("top", 0.0)]
    if quads:
        return [F.Dirichlet("inlet", h["wall"]), F.Neumann("outlet", 0.0), F.Dirichlet("bottom", 0.0),
                F.Dirichlet("top", 0.0)]
    return [F.Dirichlet("left", h["wall"]), F.Neumann("right", 0.0), F.Dirichlet("bottom", 0.0),
            F.Dirichlet("top", 0.0)]


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng([seed, 3])
    if kind == "batch":
        meshes = _batch_models(case["count"], case["lo"], case["hi"], case["pick"])
        models, prefs = [], []
        for k, mesh in enumerate(meshes):
            nu = 1.0 / float(np.exp(rng.uniform(np.log(100.0), np.log(1000.0))))
            models.append(_cavity(mesh, 1.0, nu) if k % 2 == 0 else _channel(mesh, 1.0, nu))
            prefs.append(0.0 if k % 2 == 0 else None)
            _perturb(models[-1], rng, 0.02)
        sim = F.BatchSimulation(models, _config(case), prefs, conv_break=0.0)
        return {"sim": sim, "n": 1, "fields": ("Ux", "Uy", "p"), "out": _host_fields(sim, ("Ux", "Uy", "p"))}
    mesh = _mesh_of(case)
    if kind == "simple":
        if case["mesh"] == "cavity":
            model, pref = _cavity(mesh, float(rng.uniform(0.9, 1.1)), 0.01), 0.0
            _perturb(model, rng, 0.02)
        else:
            model = _channel(mesh, float(rng.uniform(0.45, 0.55)), 1e-5, walls=("step", "bottom", "top"))
            pref = None
            _perturb(model, rng, 0.01)
        if case["mesh"] == "cavity" and case["iterations"] > 100:  # the whole run, set-up to write-back
            U = [model.U.x.values.copy(), model.U.y.values.copy()]
            return {"model": model, "config": _config(case, iterations=case["iterations"]), "pref": pref, "U": U}
        sim = F.Simulation(model, _config(case), pref, conv_break=0.0)
        return {"sim": sim, "n": case["iterations"], "fields": ("Ux", "Uy", "p"),
                "out": _host_fields(sim, ("Ux", "Uy", "p"))}
    if kind == "komega":
        model = _plate(mesh, float(rng.uniform(9.0, 11.0)))
        sim = F.Simulation(model, _config(case, turbulent=True), None, conv_break=0.0)
        names = ("Ux", "Uy", "p", "k", "omega")
        return {"sim": sim, "n": case["iterations"], "fields": names, "out": _host_fields(sim, names)}
    h = _host_inputs(case, mesh, seed)
    n, nf = mesh.ncells, mesh.nfaces
    if kind == "gradient":
        eq = {"mesh": mesh, "scheme": GRADIENT[case["scheme"]], "phi": _dev(h["phi"])}
        eq["phif"] = torch.zeros(nf, dtype=torch.float64, device="cuda")
        eq["g"] = [torch.zeros(n, dtype=torch.float64, device="cuda") for _ in range(3)]
        bcs = _bcs(case, mesh, h)
        eq["bcs"] = (L.BC * len(bcs))()
        for t, bc in zip(eq["bcs"], bcs):
            t.kind, t.patch = bc.kind, mesh.boundary_index(bc.ID)
            t.value[0] = float(bc.value)
        torch.cuda.synchronize()
        return eq
    s = {"x0": _dev(h["x0"]), "gamma": _dev(h["gamma"]), "source": _dev(h["source"])}
    phi = s["x0"].clone()
    if kind == "pressure":
        ones = torch.ones(nf, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        lap = lambda flux: [(L.OP_LAPLACIAN, F.Linear, 1, flux)]  # noqa: E731
        eq = _Equation(mesh, lap(s["gamma"]), s["source"], _bcs(case, mesh, h), phi)
        eq.precond(PRECOND[case["precond"]])
        if case["precond"] == "ldl":  # factored once, from the set-up matrix (coefficient 1), as the reference does
            gamma, eq.terms[0].flux = eq.terms[0].flux, ones.data_ptr()
            eq.discretise()
            eq.update()
            eq.terms[0].flux = gamma
        s.update(eq=eq, cfg=_solver_cfg(case, case["solver"], case["precond"]))
        return s
    s["mdot"] = _dev(h["mdot"])
    torch.cuda.synchronize()
    div = DIVERGENCE[case.get("divergence", "upwind")]
    eq = _Equation(mesh, [(L.OP_DIVERGENCE, div, 1, s["mdot"]), (L.OP_LAPLACIAN, F.Linear, -1, s["gamma"])],
                   s["source"], _bcs(case, mesh, h), phi)
    s["eq"] = eq
    if kind == "transport":
        eq.precond(F.DILU)
        s["cfg"] = _solver_cfg(case, "bicgstab", "dilu")
    return s


def _host_fields(sim, names):
    return {q: np.zeros(sim.get(q).size) for q in names}


def run(state):
    if "model" in state:  # simple(model, config): set-up, iterations, fields written back
        model = state["model"]
        model.U.x.values[:], model.U.y.values[:] = state["U"]
        model.p.values[:] = 0.0
        R = F.simple(model, state["config"], pref=state["pref"], conv_break=0.0)
        return {"Ux": model.U.x.values.copy(), "Uy": model.U.y.values.copy(), "p": model.p.values.copy(),
                "residuals": np.stack(R)}
    if "sim" in state:  # more iterations of a running simulation, then its fields on the host
        sim = state["sim"]
        sim.run(state["n"])
        for name, out in state["out"].items():
            ln = C.c_int64()
            L.check(L.lib().fvh_sim_get(sim.h, name.encode(), L.dptr(out), C.byref(ln)), "fvh_sim_get")
        return dict(state["out"])
    if "g" in state:
        g = state["g"]
        L.check(L.lib().fvh_grad(state["mesh"].device().h, state["scheme"], state["bcs"], len(state["bcs"]), 0,
                                 _p(state["phi"]), _p(state["phif"]), *(_p(t) for t in g)), "fvh_grad")
        return {"phif": state["phif"], "x": g[0], "y": g[1], "z": g[2]}
    eq = state["eq"]
    eq.discretise()
    if "cfg" not in state:
        return {"A": eq.nz, "b": eq.b}
    if "mdot" in state:  # under-relaxed, as the loops relax their transport equations
        L.check(L.lib().fvh_implicit_relax(eq.h, _p(state["x0"]), RELAX), "fvh_implicit_relax")
    eq.update()
    _copy(eq.phi, state["x0"])
    eq.solve(state["cfg"])
    return {"phi": eq.phi, "A": eq.nz, "b": eq.b}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _counts(case):
    """Cells, internal faces, matrix entries (estimates from the sizes alone)."""
    n = _cells(case)
    nif = (3 * n) // 2 if "points" in case else 2 * n
    return n, nif, n + 2 * nif


def _sweep_work(n, nnz, v):
    """One DILU-like apply: the off-diagonals, the pivots in each sweep, vectors in and out."""
    return (nnz - n) * (v + 4) + 2 * n * v + 4 * n * v


def work(case):
    n, nif, nnz = _counts(case)
    kind = case["kind"]
    v = 4 if case.get("precision") == "mixed" else 8
    spmv = nnz * (v + 4) + 2 * n * v
    asm = nif * (2 * 4 + 5 * 8) + 8 * nnz + 4 * 8 * n
    if kind == "gradient":
        passes = 3 if case["scheme"] == "midpoint" else 1
        return {"bytes": float(passes * (8 * n + 4 * 8 * nif + 2 * 4 * nif + 8 * nif + 4 * 8 * n)),
                "flops": float(passes * (4 * nif + 12 * nif))}
    if kind == "assemble":
        return {"bytes": float(asm), "flops": float(20 * nif + 10 * n)}
    if kind in ("transport", "pressure"):
        solver, pre = case.get("solver", "bicgstab"), case.get("precond", "dilu")
        apply = {"jacobi": 3 * n * v, "dilu": _sweep_work(n, nnz, v), "ilu0": _sweep_work(n, nnz, v),
                 "ldl": 2 * (12 * int(4 * n * max(1.0, np.log2(n) - 6)) + 4 * 8 * n)}[pre]
        it = case["itmax"]
        per = {"cg": spmv + apply + 10 * n * v, "bicgstab": 2 * (spmv + apply) + 20 * n * v,
               "gmres": spmv + apply + (it + 3) * 2 * n * v}[solver]
        flops = {"cg": 2 * nnz * 2 + 10 * n, "bicgstab": 8 * nnz + 20 * n, "gmres": 4 * nnz + 2 * (it + 1) * n}[solver]
        return {"bytes": float(asm + it * per), "flops": float(it * flops + 20 * nif)}
    # an iteration: two momentum solves of about two BiCGSTAB iterations, one pressure solve of 100 CG iterations
    its = case.get("iterations", 1)
    cg = 100 * (spmv + _sweep_work(n, nnz, v) + 10 * n * v)
    mom = 2 * 2 * (2 * (spmv + _sweep_work(n, nnz, v)) + 20 * n * v)
    extra = 6 * (spmv + _sweep_work(n, nnz, 8)) if kind == "komega" else 0
    return {"bytes": float(its * (cg + mom + extra + 3 * asm + 30 * 8 * n)),
            "flops": float(its * (100 * (4 * nnz + 10 * n) + 4 * (8 * nnz + 20 * n)))}


# Four times the largest difference seen: of single operators and solves against exact() over the drawn
# ranges; of whole calls against themselves with the initial velocity changed in its last place (FP64) or
# by 1e-8 (mixed), which is how far a change of rounding travels through the Krylov solves of a pass.
_TOLERANCE = {
    ("simple cavity", "fp64"): (4e-12, 4e-10), ("simple cavity", "mixed"): (1e-4, 1e-3),
    ("simple step", "fp64"): (6e-5, 3e-3), ("simple step", "mixed"): (3e-2, 0.99),
    ("komega", "fp64"): (2e-10, 1e-9), ("komega", "mixed"): (4e-3, 0.15),
    ("batch", "fp64"): (1e-10, 2e-8), ("batch", "mixed"): (1.5e-3, 0.25),
    ("transport", "fp64"): (5e-14, 1e-12), ("transport", "mixed"): (1e-6, 4e-5),
    ("pressure cg", "fp64"): (6e-12, 1e-11), ("pressure cg", "mixed"): (4e-4, 5e-3),
    ("pressure gmres", "fp64"): (6e-12, 1e-11), ("pressure gmres", "mixed"): (4e-4, 5e-3),
    ("pressure bicgstab", "fp64"): (4e-8, 4e-7), ("pressure bicgstab", "mixed"): (4e-4, 5e-3),
}


def tolerance(case):
    kind = case["kind"]
    if kind in ("assemble", "gradient"):
        return {"rel": 1e-15}
    if kind in ("simple", "pressure"):
        kind += " " + case["mesh" if kind == "simple" else "solver"]
    rel, most = _TOLERANCE[kind, case["precision"]]
    return {"rel": rel, "max": most}


# ---------------------------------------------------------------------------
# The same in plain numpy, 64 bits
# ---------------------------------------------------------------------------
class _Csr:
    """A matrix on the mesh's pattern (rows sorted by column) and its triangular-solve levels."""

    def __init__(self, mesh):
        n, fo = mesh.ncells, mesh.face_owners[mesh.nbfaces:]
        row = np.concatenate([np.arange(n), fo[:, 0], fo[:, 1]])
        col = np.concatenate([np.arange(n), fo[:, 1], fo[:, 0]])
        order = np.lexsort((col, row))
        slot = np.empty(order.size, np.int64)
        slot[order] = np.arange(order.size)
        nif = fo.shape[0]
        self.n, self.row, self.col = n, row[order], col[order]
        self.diag, self.on, self.no = slot[:n], slot[n:n + nif], slot[n + nif:]
        self.ptr = np.searchsorted(self.row, np.arange(n + 1))

    def mul(self, val, x):
        return np.bincount(self.row, val * x[self.col], minlength=self.n)

    @functools.cached_property
    def levels(self):
        """Rows by level of the forward and the backward sweep, each with its off-diagonal entries."""
        out = []
        for lower in (True, False):
            lev = np.zeros(self.n, np.int64)
            ptr, col, dg = self.ptr.tolist(), self.col.tolist(), self.diag.tolist()
            lv = lev.tolist()
            for i in (range(self.n) if lower else range(self.n - 1, -1, -1)):
                s, e = (ptr[i], dg[i]) if lower else (dg[i] + 1, ptr[i + 1])
                if e > s:
                    lv[i] = 1 + max(lv[c] for c in col[s:e])
            lev = np.array(lv)
            keep = np.nonzero(self.col < self.row if lower else self.col > self.row)[0]
            keep = keep[np.argsort(lev[self.row[keep]], kind="stable")]
            cut = np.searchsorted(lev[self.row[keep]], np.arange(1, lev.max() + 2))
            out.append([keep[a:b] for a, b in zip(cut[:-1], cut[1:])])
        return out


def _assembled(mesh, csr, terms, source, bcs):
    """A (CSR values) and b of the terms, as the finite-volume operators define them."""
    nb = mesh.nbfaces
    fo = mesh.face_owners[nb:]
    val, b = np.zeros(csr.row.size), source * mesh.cell_volume
    sgn = np.zeros(mesh.nfaces - nb)
    first = np.full(mesh.nfaces, -1.0)
    cells = np.repeat(np.arange(mesh.ncells), mesh.cell_faces_range[:, 1] - mesh.cell_faces_range[:, 0] + 1)
    own = mesh.face_owners[mesh.cell_faces, 0] == cells
    first[mesh.cell_faces[own]] = mesh.cell_nsign[own]
    sgn = first[nb:]
    for op, scheme, sign, flux in terms:
        f = flux[nb:]
        if op == L.OP_LAPLACIAN:
            ap = sign * (-f * mesh.face_area[nb:]) / mesh.face_delta[nb:]
            do, dn, oo, on = ap, ap, -ap, -ap
        else:
            ao, an = sign * f * sgn, -sign * f * sgn
            if scheme == F.Upwind:
                do, dn = np.maximum(ao, 0), np.maximum(an, 0)
                oo, on = -np.maximum(-ao, 0), -np.maximum(-an, 0)
            else:
                return None  # the linear weights belong to the mesh builder
        val[csr.on] += oo
        val[csr.no] += on
        val[csr.diag] += np.bincount(fo[:, 0], do, minlength=csr.n) + np.bincount(fo[:, 1], dn, minlength=csr.n)
        for bc in bcs:
            fs, cs = mesh.boundary(bc.ID)
            if op == L.OP_LAPLACIAN and bc.kind == L.BC_DIRICHLET:
                ap = -sign * flux[fs] * mesh.face_area[fs] / mesh.face_delta[fs]
                np.add.at(val, csr.diag[cs], ap)
                np.add.at(b, cs, ap * bc.value)
            elif op == L.OP_DIVERGENCE:
                ap = sign * flux[fs]
                if bc.kind == L.BC_DIRICHLET:
                    np.add.at(b, cs, -ap * bc.value)
                else:
                    np.add.at(val, csr.diag[cs], np.maximum(ap, 0))
    return val, b


def _transposed(csr):
    """Per entry (i, j) the slot of (j, i)."""
    t = np.arange(csr.row.size)
    t[csr.on], t[csr.no] = csr.no, csr.on
    return t


def _dilu(csr, val):
    """x -> M^-1 x with M = (D + L) D^-1 (D + U)."""
    fwd, bwd = csr.levels
    D, t = val[csr.diag].copy(), _transposed(csr)
    for e in fwd:
        np.subtract.at(D, csr.row[e], val[e] * val[t[e]] / D[csr.col[e]])

    def apply(x):
        y = x.copy()
        for e in fwd:
            np.subtract.at(y, csr.row[e], val[e] * y[csr.col[e]] / D[csr.col[e]])
        z = y / D
        for e in bwd:
            np.subtract.at(z, csr.row[e], val[e] * z[csr.col[e]] / D[csr.row[e]])
        return z

    return apply


def _ilu0(csr, val, nx):
    """x -> (LU)^-1 x of ILU(0) on a five-point grid (no fill meets the pattern off the diagonal)."""
    fwd, bwd = csr.levels
    lu, t = val.copy(), _transposed(csr)
    for e in fwd:
        lu[e] = val[e] / lu[csr.diag[csr.col[e]]]
        np.subtract.at(lu, csr.diag[csr.row[e]], lu[e] * val[t[e]])

    def apply(x):
        y = x.copy()
        for e in fwd:
            np.subtract.at(y, csr.row[e], lu[e] * y[csr.col[e]])
        d = lu[csr.diag]
        z = y / d
        for e in bwd:
            np.subtract.at(z, csr.row[e], lu[e] * z[csr.col[e]] / d[csr.row[e]])
        return z

    return apply


def _direct(csr, val, nx, ny):
    """x -> A^-1 x by block elimination over the columns of an nx x ny grid."""
    i, j = csr.row % nx, csr.row // nx
    ci, cj = csr.col % nx, csr.col // nx
    T = np.zeros((nx, ny, ny))
    same, right, left = ci == i, ci == i + 1, ci == i - 1
    T[i[same], j[same], cj[same]] = val[same]
    up, lo = np.zeros((nx, ny)), np.zeros((nx, ny))
    up[i[right], j[right]] = val[right]
    lo[i[left], j[left]] = val[left]
    inv = []
    S = T[0]
    for k in range(nx):
        if k:
            S = T[k] - lo[k][:, None] * inv[-1] * up[k - 1][None, :]
        inv.append(np.linalg.inv(S))

    def apply(x):
        g = x.reshape(ny, nx).T.copy()
        for k in range(1, nx):
            g[k] -= lo[k] * (inv[k - 1] @ g[k - 1])
        z = np.empty_like(g)
        z[-1] = inv[-1] @ g[-1]
        for k in range(nx - 2, -1, -1):
            z[k] = inv[k] @ (g[k] - up[k] * z[k + 1])
        return z.T.reshape(-1)

    return apply


def _bicgstab(mul, M, b, x0, itmax):
    """Left-preconditioned, shadow residual b."""
    x, r = np.zeros_like(b), M(b - mul(x0))
    p, rho = r.copy(), b @ r
    for _ in range(itmax):
        v = M(mul(p))
        alpha = rho / (b @ v)
        s = r - alpha * v
        x += alpha * p
        t = M(mul(s))
        omega = (t @ s) / (t @ t)
        x += omega * s
        r = s - omega * t
        nxt = b @ r
        p = r + (nxt / rho) * (alpha / omega) * (p - omega * v)
        rho = nxt
    return x + x0


def _cg(mul, M, b, x0, itmax):
    x, r = np.zeros_like(b), b - mul(x0)
    z = M(r)
    p, gamma = z.copy(), r @ z
    for _ in range(itmax):
        Ap = mul(p)
        alpha = gamma / (p @ Ap)
        x += alpha * p
        r = r - alpha * Ap
        z = M(r)
        nxt = r @ z
        p = z + (nxt / gamma) * p
        gamma = nxt
    return x + x0


def _gmres(mul, M, b, x0, itmax):
    r = M(b - mul(x0))
    V, H = [r / np.linalg.norm(r)], np.zeros((itmax + 1, itmax))
    for k in range(itmax):
        q = M(mul(V[k]))
        for i in range(k + 1):
            H[i, k] = V[i] @ q
            q = q - H[i, k] * V[i]
        H[k + 1, k] = np.linalg.norm(q)
        V.append(q / H[k + 1, k])
    e = np.zeros(itmax + 1)
    e[0] = np.linalg.norm(r)
    y = np.linalg.lstsq(H, e, rcond=None)[0]
    return x0 + np.array(V[:itmax]).T @ y


def _gradient(mesh, scheme, phi, bcs):
    nb, o1, o2 = mesh.nbfaces, mesh.face_owners[:, 0], mesh.face_owners[:, 1]
    S = mesh.face_area[:, None] * mesh.face_normal
    w = mesh.face_weight if scheme == F.Orthogonal else np.full(mesh.nfaces, 0.5)
    phif = w * phi[o1] + (1 - w) * phi[o2]
    for bc in bcs:
        fs, cs = mesh.boundary(bc.ID)
        phif[fs] = bc.value if bc.kind == L.BC_DIRICHLET else phi[cs]
    cells = np.repeat(np.arange(mesh.ncells), mesh.cell_faces_range[:, 1] - mesh.cell_faces_range[:, 0] + 1)
    cf, ns = mesh.cell_faces, mesh.cell_nsign

    def gauss():
        g = []
        for d in range(3):
            a = np.bincount(cells, phif[cf] * S[cf, d] * ns, minlength=mesh.ncells)
            a += np.bincount(o1[:nb], phif[:nb] * S[:nb, d], minlength=mesh.ncells)
            g.append(a / mesh.cell_volume)
        return g

    g = gauss()
    if scheme == F.Midpoint:
        a, c = o1[nb:], o2[nb:]
        arm = mesh.face_centre[nb:] - 0.5 * (mesh.cell_centre[a] + mesh.cell_centre[c])
        for _ in range(2):
            phif[nb:] = 0.5 * (phi[a] + phi[c]) + sum(0.5 * (g[d][a] + g[d][c]) * arm[:, d] for d in range(3))
            g = gauss()
    return {"phif": phif, "x": g[0], "y": g[1], "z": g[2]}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("simple", "komega", "batch"):
        return None  # numpy takes minutes for the sweeps of that many Krylov iterations
    mesh = _mesh_of(case)
    h = _host_inputs(case, mesh, seed)
    bcs = _bcs(case, mesh, h)
    if kind == "gradient":
        return _gradient(mesh, GRADIENT[case["scheme"]], h["phi"], bcs)
    csr = _Csr(mesh)
    if kind == "pressure":
        terms = [(L.OP_LAPLACIAN, F.Linear, 1, h["gamma"])]
    else:
        terms = [(L.OP_DIVERGENCE, DIVERGENCE[case.get("divergence", "upwind")], 1, h["mdot"]),
                 (L.OP_LAPLACIAN, F.Linear, -1, h["gamma"])]
    got = _assembled(mesh, csr, terms, h["source"], bcs)
    if got is None:
        return None
    val, b = got
    if kind == "assemble":
        return {"A": val, "b": b}
    if kind == "transport":
        val[csr.diag] /= RELAX
        b = b + (1.0 - RELAX) * val[csr.diag] * h["x0"]
    pre, solver, itmax = case.get("precond", "dilu"), case.get("solver", "bicgstab"), case["itmax"]
    cost = itmax * (2 if solver == "bicgstab" else 1) * mesh.ncells * {"jacobi": 0.1, "ldl": 0.3}.get(pre, 1.0)
    if cost > 4e6:
        return None  # over 20 seconds
    if pre == "ldl":
        setup, _ = _assembled(mesh, csr, [(L.OP_LAPLACIAN, F.Linear, 1, np.ones(mesh.nfaces))], h["source"], bcs)
        M = _direct(csr, setup, case["nx"], case["ny"])
    elif pre == "jacobi":
        scale = 1.0 / np.abs(val[csr.diag])
        M = lambda x: scale * x  # noqa: E731
    else:
        M = _dilu(csr, val) if pre == "dilu" else _ilu0(csr, val, case.get("nx"))
    solve = {"cg": _cg, "bicgstab": _bicgstab, "gmres": _gmres}[solver]
    mul = lambda x: csr.mul(val, x)  # noqa: E731
    x0 = h["x0"]
    if case["precision"] == "mixed":  # defect correction: the inner solve starts from 0 on the defect
        phi = x0 + solve(mul, M, b - mul(x0), np.zeros_like(b), itmax)
    else:
        phi = solve(mul, M, b, x0, itmax)
    return {"phi": phi, "A": val, "b": b}
