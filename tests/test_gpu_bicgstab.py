"""BiCGSTAB's fused launches against the oracle, bit for bit: banded and
general rows, with and without the sweeps' layout, one chunk and several, more
rows than the fused grids have threads, and every end of the iteration."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from oracle import ref
from tests.cases import same_bits

pytestmark = pytest.mark.gpu
LIB = L.lib

MESHES = {"row": lambda: F.channel(7, 1), "column": lambda: F.channel(1, 2049), "two chunks": lambda: F.channel(64, 33),
          "more rows than threads": lambda: F.channel(700, 400), "triangles": lambda: F.delaunay_unit_square(1500, seed=4)}


@pytest.mark.parametrize("mesh", list(MESHES))
@pytest.mark.parametrize("precond", [L.PRECOND_DILU, L.PRECOND_JACOBI, L.PRECOND_NONE])
def test_bicgstab_against_the_oracle(mesh, precond):
    mesh = MESHES[mesh]()
    dm = mesh.device()
    rp, ci = dm.pattern()
    n = mesh.ncells
    rng = np.random.default_rng(n)
    rows = np.repeat(np.arange(n), np.diff(rp))
    vals = np.where(rows == ci, 4.4 + rng.random(ci.size), -0.5 - 0.6 * rng.random(ci.size))
    b, x = rng.standard_normal(n), rng.standard_normal(n)
    eq, nz, rhs = C.c_void_p(), C.c_void_p(), C.c_void_p()
    L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
    try:
        L.check(LIB().fvh_eqn_arrays(eq, C.byref(nz), C.byref(rhs)))
        L.check(LIB().fvh_memcpy(nz, vals.ctypes.data_as(C.c_void_p), vals.nbytes))
        L.check(LIB().fvh_precond_set(eq, precond, None))
        L.check(LIB().fvh_precond_update(eq))
        for bscale, itmax, rtol in ((1.0, 30, 1e-9), (1.0, 1, 1e-9), (1.0, 2, 0.0), (1.0, 7, 0.0), (0.0, 9, 1e-9)):
            bb, x0 = bscale * b, (bscale != 0.0) * 0.1 * x
            L.check(LIB().fvh_memcpy(rhs, bb.ctypes.data_as(C.c_void_p), bb.nbytes))
            cfg = L.SolverCfg(solver=L.BICGSTAB, precond=precond, itmax=itmax, precision=L.FP64, convergence=0.0,
                              relax=1.0, atol=0.0, rtol=rtol)
            st, phi = L.Stats(), L.DeviceArray.from_host(x0)
            L.check(LIB().fvh_solve(eq, C.byref(cfg), phi.vp, C.byref(st)), "fvh_solve")
            want, wst, _ = ref.solve_csr(mesh, vals, bb, cfg, x0)
            assert st.niter == wst["niter"], (bscale, itmax, rtol)
            assert L.KRYLOV_STATUS.get(st.status, st.status) == wst["status"], (bscale, itmax, rtol)
            assert same_bits(phi.host(), want) and same_bits(st.rnorm, wst["rnorm"]), (bscale, itmax, rtol)
    finally:
        LIB().fvh_eqn_destroy(eq)


@pytest.mark.parametrize("size", [(65, 33), (130, 64), (700, 400)])
@pytest.mark.parametrize("precond", [L.PRECOND_DILU, L.PRECOND_ILU0, L.PRECOND_JACOBI, L.PRECOND_NONE])
def test_fused_fp32_inner_solves(size, precond, monkeypatch):
    """The FP32 solves inside the FP64 correction, with the products in the
    sweeps' layout (or by band position) and in natural CSR rows: the same bits
    where both apply one arithmetic (ILU(0)'s differs by walk).  Both reach
    the FP64 solve's residual past the FP32 limit in a like number of iterations."""
    got = {}
    for sweep in ("band", "levels"):
        if sweep == "levels":
            monkeypatch.setenv("FVH_SWEEP", "levels")
        else:
            monkeypatch.delenv("FVH_SWEEP", raising=False)
        mesh = F.channel(*size)
        dm = mesh.device()
        rp, ci = dm.pattern()
        n = mesh.ncells
        rng = np.random.default_rng(n)
        rows = np.repeat(np.arange(n), np.diff(rp))
        vals = np.where(rows == ci, 4.4 + rng.random(ci.size), -0.5 - 0.6 * rng.random(ci.size))
        b, x = rng.standard_normal(n), 0.1 * rng.standard_normal(n)
        defect = lambda y: np.linalg.norm(b - np.bincount(rows, vals * y[ci], n))  # noqa: E731
        eq, nz, rhs = C.c_void_p(), C.c_void_p(), C.c_void_p()
        L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
        try:
            L.check(LIB().fvh_eqn_arrays(eq, C.byref(nz), C.byref(rhs)))
            L.check(LIB().fvh_memcpy(nz, vals.ctypes.data_as(C.c_void_p), vals.nbytes))
            L.check(LIB().fvh_memcpy(rhs, b.ctypes.data_as(C.c_void_p), b.nbytes))
            L.check(LIB().fvh_precond_set(eq, precond, None))
            L.check(LIB().fvh_precond_update(eq))
            its = {}
            for precision, itmax, rtol in ((L.FP64, 200, 1e-9), (L.MIXED, 200, 1e-9), (L.MIXED, 1, 1e-4),
                                           (L.MIXED, 2, 1e-4), (L.MIXED, 7, 1e-4)):
                cfg = L.SolverCfg(solver=L.BICGSTAB, precond=precond, itmax=itmax, precision=precision,
                                  convergence=0.0, relax=1.0, atol=0.0, rtol=rtol)
                st, phi = L.Stats(), L.DeviceArray.from_host(x)
                L.check(LIB().fvh_solve(eq, C.byref(cfg), phi.vp, C.byref(st)), "fvh_solve")
                y = phi.host()
                if itmax == 200:
                    its[precision] = st.niter
                    # the residual that stops FP64 is the preconditioned one
                    assert defect(y) <= 1e-8 * defect(x), (sweep, precision, defect(y) / defect(x))
                if precision == L.MIXED:
                    got[sweep, itmax] = np.append(y, [st.niter, st.status, st.rnorm])
            # a restart of the Krylov space at each of the few corrections
            assert its[L.MIXED] <= 2 * its[L.FP64] + 4, its
        finally:
            LIB().fvh_eqn_destroy(eq)
    if precond != L.PRECOND_ILU0:
        for itmax in (200, 1, 2, 7):
            assert same_bits(got["band", itmax], got["levels", itmax]), itmax
