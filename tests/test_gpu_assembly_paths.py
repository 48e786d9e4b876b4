"""The partial modes of the assembly touch only the cells they change: the
reference value its cell, boundary conditions the cells of their patches.
Expected values by hand on the assembled arrays, bit for bit."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from oracle import ref
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


def _both(spec):
    """A term list for the device and for the oracle: (operator, scheme, sign, flux, phi)."""
    dev, host, keep = (L.Term * len(spec))(), (L.Term * len(spec))(), []
    for k, (op, scheme, sign, *fields) in enumerate(spec):
        for t in (dev[k], host[k]):
            t.op, t.scheme, t.sign = op, scheme, sign
        for attr, a in zip(("flux", "phi"), fields):
            if a is not None:
                d, h = L.DeviceArray.from_host(a), np.ascontiguousarray(a)
                keep += [d, h]
                setattr(dev[k], attr, d.ptr)
                setattr(host[k], attr, h.ctypes.data)
    return dev, host, keep


@pytest.mark.parametrize("nx,ny", [(1, 1), (2, 1), (16, 16), (257, 3)])
def test_a_new_term_list_replaces_the_whole_matrix(nx, ny):
    """discretise! zeroes A first: an equation assembled before keeps nothing of
    it, whatever the next model's terms (none of a face among them)."""
    mesh = F.channel(nx, ny)
    dm = mesh.device()
    n, nf = mesh.ncells, mesh.nfaces
    rng = np.random.default_rng(n)
    flux, gam, si, prev = rng.standard_normal(nf), 1.0 + rng.random(nf), rng.random(n), rng.standard_normal(n)
    face = [(L.OP_DIVERGENCE, F.Upwind, 1, flux, None), (L.OP_LAPLACIAN, F.Linear, -1, gam, None)]
    time, source = [(L.OP_TIME, F.Euler, 1, None, None)], [(L.OP_SI, F.Linear, -1, si, prev)]
    steady = [(L.OP_TIME, F.Steady, 1, None, None)]
    dprev, eq = L.DeviceArray.from_host(prev), C.c_void_p()
    none = (L.BC * 1)()
    L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
    try:
        for spec in (face, time, face + time, source, face[:1], steady, face[1:] + source, time + source):
            dev, host, keep = _both(spec)
            L.check(LIB().fvh_discretise(eq, dev, len(spec), None, 0, dprev.vp, 0.25))
            gA, gb = _arrays(eq, dm.pattern()[1].size, n)
            A, b = ref.assemble(mesh, host, len(spec), None, 0, prev, 0.25, none, 0, 0)
            assert same_bits(gA, A) and same_bits(gb, b), (nx, ny, [t[0] for t in spec])
    finally:
        LIB().fvh_eqn_destroy(eq)
