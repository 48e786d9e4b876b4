"""The partial modes of the assembly touch only the cells they change: the
reference value its cell, boundary conditions the cells of their patches.
Expected values by hand on the assembled arrays, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from tests.cases import same_bits

pytestmark = pytest.mark.gpu
LIB = L.lib


def _arrays(eq, nnz, n):
    nz, b = C.c_void_p(), C.c_void_p()
    L.check(LIB().fvh_eqn_arrays(eq, C.byref(nz), C.byref(b)))
    A, rhs = np.zeros(nnz), np.zeros(n)
    L.check(LIB().fvh_memcpy(A.ctypes.data_as(C.c_void_p), nz, A.nbytes))
    L.check(LIB().fvh_memcpy(rhs.ctypes.data_as(C.c_void_p), b, rhs.nbytes))
    return A, rhs


@pytest.mark.parametrize("nx,ny", [(1, 1), (2, 1), (1, 9), (16, 16), (257, 3)])
def test_reference_and_boundary_passes(nx, ny):
    mesh = F.channel(nx, ny)
    dm = mesh.device()
    rp, ci = dm.pattern()
    n, diag = mesh.ncells, np.zeros(mesh.ncells, np.int64)
    rows = np.repeat(np.arange(n), np.diff(rp))
    diag[rows[rows == ci]] = np.nonzero(rows == ci)[0]
    gam = L.DeviceArray.from_host(1.0 + 0.1 * np.arange(mesh.nfaces))
    terms = (L.Term * 1)()
    terms[0].op, terms[0].scheme, terms[0].sign, terms[0].flux = L.OP_LAPLACIAN, F.Linear, 1, gam.ptr
    for cell in sorted({0, n // 2, n - 1}):
        eq = C.c_void_p()
        L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
        try:
            L.check(LIB().fvh_discretise(eq, terms, 1, None, 0, None, 1.0))
            A, b = _arrays(eq, ci.size, n)
            # a corner cell has faces of several patches: entries in BC order
            bcs = [F.Dirichlet("top", 2.0), F.Neumann("inlet", 0.0), F.Dirichlet("outlet", 3.0)]
            arr = F.api._bcs(mesh, bcs, False)
            L.check(LIB().fvh_apply_bcs(eq, terms, 1, arr, len(bcs), 0))
            for bc in bcs:
                for f, c in zip(*mesh.boundary(bc.ID)):
                    if bc.kind == L.BC_DIRICHLET:
                        ap = -((1.0 + 0.1 * f) * mesh.face_area[f] / mesh.face_delta[f])
                        A[diag[c]] += ap
                        b[c] += ap * bc.value
            L.check(LIB().fvh_set_reference(eq, 0.75, cell))
            b[cell] += A[diag[cell]] * 0.75
            A[diag[cell]] += A[diag[cell]]
            gA, gb = _arrays(eq, ci.size, n)
            assert same_bits(gA, A) and same_bits(gb, b), (nx, ny, cell)
        finally:
            LIB().fvh_eqn_destroy(eq)
