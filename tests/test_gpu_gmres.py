"""GMRES's Gram-Schmidt steps (each forming its own coefficient) against the
oracle, bit for bit, one row either side of the 2,048-row chunks of the
sums, for one basis vector and many."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from oracle import ref
from tests.cases import same_bits

pytestmark = pytest.mark.gpu
LIB = L.lib


@pytest.mark.parametrize("nx,ny", [(2, 1), (89, 23), (64, 32), (3, 683), (17, 241), (130, 65)])
@pytest.mark.parametrize("precond", [L.PRECOND_DILU, L.PRECOND_JACOBI, L.PRECOND_NONE])
def test_gmres_against_the_oracle(nx, ny, precond):
    mesh = F.channel(nx, ny)
    dm = mesh.device()
    rp, ci = dm.pattern()
    n = mesh.ncells
    rng = np.random.default_rng(n)
    rows = np.repeat(np.arange(n), np.diff(rp))
    vals = np.where(rows == ci, 4.4 + rng.random(ci.size), -0.5 - 0.6 * rng.random(ci.size))
    b, x = rng.standard_normal(n), 0.1 * rng.standard_normal(n)
    eq, nz, rhs = C.c_void_p(), C.c_void_p(), C.c_void_p()
    L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
    try:
        L.check(LIB().fvh_eqn_arrays(eq, C.byref(nz), C.byref(rhs)))
        L.check(LIB().fvh_memcpy(nz, vals.ctypes.data_as(C.c_void_p), vals.nbytes))
        L.check(LIB().fvh_memcpy(rhs, b.ctypes.data_as(C.c_void_p), b.nbytes))
        L.check(LIB().fvh_precond_set(eq, precond, None))
        L.check(LIB().fvh_precond_update(eq))
        for itmax, rtol in ((40, 1e-9), (1, 1e-9), (2, 0.0), (11, 0.0)):
            cfg = L.SolverCfg(solver=L.GMRES, precond=precond, itmax=itmax, precision=L.FP64, convergence=0.0,
                              relax=1.0, atol=0.0, rtol=rtol)
            st, phi = L.Stats(), L.DeviceArray.from_host(x)
            L.check(LIB().fvh_solve(eq, C.byref(cfg), phi.vp, C.byref(st)), "fvh_solve")
            want, wst, _ = ref.solve_csr(mesh, vals, b, cfg, x)
            assert st.niter == wst["niter"], (itmax, rtol)
            assert L.KRYLOV_STATUS.get(st.status, st.status) == wst["status"], (itmax, rtol)
            assert same_bits(phi.host(), want) and same_bits(st.rnorm, wst["rnorm"]), (itmax, rtol)
    finally:
        LIB().fvh_eqn_destroy(eq)


@pytest.mark.parametrize("rows", ["band", "csr"])
@pytest.mark.parametrize("nx,ny", [(1049, 1000), (2098, 1000)])
def test_large_systems_against_the_oracle(nx, ny, rows, monkeypatch):
    """Past the rows where the updates leave BiCGSTAB's products (2^20) and where
    the vector passes and Gram-Schmidt sums change form (2^21): a few
    iterations, bit for bit."""
    if rows == "csr":
        monkeypatch.setenv("FVH_SWEEP", "levels")
    mesh = F.channel(nx, ny)
    dm = mesh.device()
    rp, ci = dm.pattern()
    n = mesh.ncells
    print(f"{nx}x{ny} {rows}", flush=True)
    rng = np.random.default_rng(n)
    on = np.repeat(np.arange(n), np.diff(rp)) == ci
    vals = np.where(on, 4.4 + rng.random(ci.size), -0.5 - 0.6 * rng.random(ci.size))
    b, x = rng.standard_normal(n), 0.1 * rng.standard_normal(n)
    eq, nz, rhs = C.c_void_p(), C.c_void_p(), C.c_void_p()
    L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
    try:
        L.check(LIB().fvh_eqn_arrays(eq, C.byref(nz), C.byref(rhs)))
        L.check(LIB().fvh_memcpy(nz, vals.ctypes.data_as(C.c_void_p), vals.nbytes))
        L.check(LIB().fvh_memcpy(rhs, b.ctypes.data_as(C.c_void_p), b.nbytes))
        L.check(LIB().fvh_precond_set(eq, L.PRECOND_JACOBI, None))
        L.check(LIB().fvh_precond_update(eq))
        for solver in (L.BICGSTAB, L.GMRES):
            cfg = L.SolverCfg(solver=solver, precond=L.PRECOND_JACOBI, itmax=3, precision=L.FP64, convergence=0.0,
                              relax=1.0, atol=0.0, rtol=0.0)
            st, phi = L.Stats(), L.DeviceArray.from_host(x)
            L.check(LIB().fvh_solve(eq, C.byref(cfg), phi.vp, C.byref(st)), "fvh_solve")
            want, wst, _ = ref.solve_csr(mesh, vals, b, cfg, x)
            assert st.niter == wst["niter"] == 3
            assert same_bits(phi.host(), want) and same_bits(st.rnorm, wst["rnorm"]), (solver, rows)
    finally:
        LIB().fvh_eqn_destroy(eq)
