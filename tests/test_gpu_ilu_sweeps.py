"""ILU(0) on the pipelined band sweeps against the level-scheduled kernels
(FVH_SWEEP=levels when the mesh is made): FP64 applies and solves bit for bit,
at the sweeps' edges (64 rows a wave, one row, one column, several blocks).
FP32 applies round differently (premultiplied coefficients, fused): both stay
within 1e-6 of the FP64 apply, a few roundings of 6e-8 for these dominant
matrices, and the sweeps' error is no larger than the level walk's (measured
0.84 to 0.91 of it above 1,000 rows)."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from tests.cases import same_bits

pytestmark = pytest.mark.gpu
LIB = L.lib


def _results(nx, ny, levels, monkeypatch):
    if levels:
        monkeypatch.setenv("FVH_SWEEP", "levels")
    else:
        monkeypatch.delenv("FVH_SWEEP", raising=False)
    mesh = F.channel(nx, ny)
    dm = mesh.device()
    rp, ci = dm.pattern()
    rng = np.random.default_rng(nx + 1000 * ny)
    rows = np.repeat(np.arange(mesh.ncells), np.diff(rp))
    vals = np.where(rows == ci, -4.2 - rng.random(ci.size), 0.7 + 0.5 * rng.random(ci.size))
    x = rng.standard_normal(mesh.ncells)
    eq, nz, b = C.c_void_p(), C.c_void_p(), C.c_void_p()
    L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
    try:
        L.check(LIB().fvh_eqn_arrays(eq, C.byref(nz), C.byref(b)))
        L.check(LIB().fvh_memcpy(nz, vals.ctypes.data_as(C.c_void_p), vals.nbytes))
        L.check(LIB().fvh_memcpy(b, x.ctypes.data_as(C.c_void_p), x.nbytes))
        L.check(LIB().fvh_precond_set(eq, L.PRECOND_ILU0, None))
        out = {}
        for k in range(2):  # a second update on the same records
            L.check(LIB().fvh_precond_update(eq))
            dx, dy = L.DeviceArray.from_host(x), L.DeviceArray(x.size)
            L.check(LIB().fvh_precond_apply(eq, dy.vp, dx.vp), "fvh_precond_apply")
            out[f"apply {k}"] = dy.host()
        fx, fy = L.DeviceArray.from_host(x.astype(np.float32)), L.DeviceArray(x.size, np.float32)
        L.check(LIB().fvh_precond_apply_f32(eq, fy.vp, fx.vp), "fvh_precond_apply_f32")
        out["f32"] = fy.host()
        for solver in (L.CG, L.BICGSTAB, L.GMRES):
            cfg = L.SolverCfg(solver=solver, precond=L.PRECOND_ILU0, itmax=12, precision=L.FP64, convergence=0.0,
                              relax=1.0, atol=0.0, rtol=1e-6)
            st, phi = L.Stats(), L.DeviceArray.from_host(0.1 * x)
            L.check(LIB().fvh_solve(eq, C.byref(cfg), phi.vp, C.byref(st)), "fvh_solve")
            out[f"solve {solver}"] = np.append(phi.host(), [st.niter, st.status, st.rnorm])
        return out
    finally:
        LIB().fvh_eqn_destroy(eq)


@pytest.mark.parametrize("nx,ny", [(7, 1), (1, 7), (3, 3), (40, 63), (40, 64), (65, 65), (130, 200), (517, 129)])
def test_ilu0_sweeps_against_levels(nx, ny, monkeypatch):
    got, want = _results(nx, ny, False, monkeypatch), _results(nx, ny, True, monkeypatch)
    for name in want:
        if name == "f32":
            ref = want["apply 0"]
            err, err0 = (np.linalg.norm(y - ref) / np.linalg.norm(ref) for y in (got[name], want[name]))
            print(f"{nx}x{ny}: FP32 error {err:.2e}, level walk {err0:.2e}")
            assert err <= 1e-6 and err0 <= 1e-6, name
            if nx * ny > 1000:
                assert err <= err0, name
        else:
            assert same_bits(got[name], want[name]), f"{nx}x{ny} {name}"
