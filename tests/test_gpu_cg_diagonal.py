"""CG with an elementwise preconditioner (applied where r is updated) against the
oracle, bit for bit: banded and general rows, one chunk and several, remainders
of a chunk, and every end of the iteration."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from oracle import ref
from tests.cases import same_bits

pytestmark = pytest.mark.gpu
LIB = L.lib

MESHES = {"one cell": lambda: F.channel(1, 1), "row": lambda: F.channel(255, 1), "a chunk": lambda: F.channel(64, 32),
          "a chunk and a row": lambda: F.channel(1, 2049), "chunks": lambda: F.channel(300, 211),
          "triangles": lambda: F.delaunay_unit_square(1500, seed=4)}


@pytest.mark.parametrize("mesh", list(MESHES))
@pytest.mark.parametrize("precond", [L.PRECOND_JACOBI, L.PRECOND_NORMDIAG, L.PRECOND_NONE])
def test_cg_against_the_oracle(mesh, precond):
    mesh = MESHES[mesh]()
    dm = mesh.device()
    rp, ci = dm.pattern()
    n = mesh.ncells
    rng = np.random.default_rng(n)
    rows = np.repeat(np.arange(n), np.diff(rp))
    w = 0.5 + 0.5 * np.sin(1.0 + 7.0 * np.minimum(rows, ci) + 3.0 * np.maximum(rows, ci)) ** 2
    vals = np.where(rows == ci, -4.1 - 0.1 * rng.random(ci.size), w)  # solved with the sign turned
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
            cfg = L.SolverCfg(solver=L.CG, precond=precond, itmax=itmax, precision=L.FP64, convergence=0.0,
                              relax=1.0, atol=0.0, rtol=rtol)
            st, phi = L.Stats(), L.DeviceArray.from_host(x0)
            L.check(LIB().fvh_solve(eq, C.byref(cfg), phi.vp, C.byref(st)), "fvh_solve")
            want, wst, _ = ref.solve_csr(mesh, vals, bb, cfg, x0)
            assert st.niter == wst["niter"], (bscale, itmax, rtol)
            assert L.KRYLOV_STATUS.get(st.status, st.status) == wst["status"], (bscale, itmax, rtol)
            assert same_bits(phi.host(), want) and same_bits(st.rnorm, wst["rnorm"]), (bscale, itmax, rtol)
    finally:
        LIB().fvh_eqn_destroy(eq)
