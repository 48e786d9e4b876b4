"""CG iterations in one work-group on small grids against the launch-by-launch
iterations (FVH_CG_FUSED=0), bit for bit: at the sweeps' edges (64 rows a wave,
one row, one column, three waves), the reduction's (2048-row chunks) and the
rule's (4096 rows, 512 steps of walk), for every end of the iteration."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from tests.cases import same_bits

pytestmark = pytest.mark.gpu
LIB = L.lib


def _solves(mesh, precond, precision, cases):
    dm = mesh.device()
    rp, ci = dm.pattern()
    n = mesh.ncells
    rng = np.random.default_rng(n)
    rows = np.repeat(np.arange(n), np.diff(rp))
    # symmetric: each coupling depends on the pair of cells alone
    lo, hi = np.minimum(rows, ci), np.maximum(rows, ci)
    w = 0.5 + 0.5 * np.sin(1.0 + 7.0 * lo + 3.0 * hi) ** 2
    vals = np.where(rows == ci, 0.0, w)
    vals[rows == ci] = -1.02 * np.bincount(rows, vals, n) - 0.01
    b, x = rng.standard_normal(n), rng.standard_normal(n)
    eq, nz, rhs = C.c_void_p(), C.c_void_p(), C.c_void_p()
    L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
    out = []
    try:
        L.check(LIB().fvh_eqn_arrays(eq, C.byref(nz), C.byref(rhs)))
        L.check(LIB().fvh_precond_set(eq, precond, None))
        for scale, bscale, itmax, rtol in cases:
            v, bb = np.ascontiguousarray(scale * vals), np.ascontiguousarray(bscale * b)
            L.check(LIB().fvh_memcpy(nz, v.ctypes.data_as(C.c_void_p), v.nbytes))
            L.check(LIB().fvh_memcpy(rhs, bb.ctypes.data_as(C.c_void_p), bb.nbytes))
            L.check(LIB().fvh_precond_update(eq))
            cfg = L.SolverCfg(solver=L.CG, precond=precond, itmax=itmax, precision=precision, convergence=0.0,
                              relax=1.0, atol=0.0, rtol=rtol)
            st, phi = L.Stats(), L.DeviceArray.from_host((bscale != 0.0) * 0.1 * x)
            L.check(LIB().fvh_solve(eq, C.byref(cfg), phi.vp, C.byref(st)), "fvh_solve")
            out.append(np.append(phi.host(), [st.niter, st.status, st.rnorm]))
        return out
    finally:
        LIB().fvh_eqn_destroy(eq)


SIZES = [(1, 1), (5, 1), (1, 7), (40, 40), (64, 63), (31, 64), (31, 65), (32, 64), (17, 127), (16, 128), (21, 190),
         (2049, 1), (409, 10), (448, 9), (449, 9), (64, 64), (4096, 1), (65, 64)]


@pytest.mark.parametrize("nx,ny", SIZES)
def test_one_work_group_cg_keeps_the_bits(nx, ny, monkeypatch):
    mesh = F.channel(nx, ny)
    # solved; out of iterations after 1, 3 and more than one launch's worth;
    # b = 0 (nothing to iterate); A = 0 would not factor: a tiny A reaches the
    # zero-curvature exit or not, alike
    cases = [(1.0, 1.0, 60, 1e-8), (1.0, 1.0, 1, 1e-8), (1.0, 1.0, 3, 0.0), (1.0, 0.0, 9, 1e-8), (1e-30, 1.0, 5, 0.0)]
    if (nx, ny) in ((40, 40), (31, 65)):
        cases.append((1.0, 1.0, 300, 0.0))
    for precond in (L.PRECOND_DILU, L.PRECOND_ILU0):
        for precision in (L.FP64, L.MIXED):
            monkeypatch.delenv("FVH_CG_FUSED", raising=False)
            got = _solves(mesh, precond, precision, cases)
            monkeypatch.setenv("FVH_CG_FUSED", "0")
            ref = _solves(mesh, precond, precision, cases)
            for case, g, r in zip(cases, got, ref):
                assert same_bits(g, r), (precond, precision, case, g[-3:], r[-3:])
