"""ILU(0) and DILU on the band sweeps keep records of their own: an update, or
a set-up, of one leaves nothing in the other's, and an update leaves nothing of
the matrix before it."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L
from tests.cases import same_bits

pytestmark = pytest.mark.gpu
LIB = L.lib


class _Eq:
    def __init__(self, dm, n):
        self.h, nz = C.c_void_p(), C.c_void_p()
        L.check(LIB().fvh_eqn_create(dm.h, C.byref(self.h)))
        L.check(LIB().fvh_eqn_arrays(self.h, C.byref(nz), None))
        self.nz, self.n = nz, n

    def __enter__(self):
        return self

    def __exit__(self, *a):
        LIB().fvh_eqn_destroy(self.h)

    def set(self, kind):
        L.check(LIB().fvh_precond_set(self.h, kind, None))

    def update(self, vals):
        L.check(LIB().fvh_memcpy(self.nz, vals.ctypes.data_as(C.c_void_p), vals.nbytes))
        L.check(LIB().fvh_precond_update(self.h))

    def apply(self, x, f32=False):
        t = np.float32 if f32 else np.float64
        dx, dy = L.DeviceArray.from_host(x.astype(t)), L.DeviceArray(self.n, t)
        L.check((LIB().fvh_precond_apply_f32 if f32 else LIB().fvh_precond_apply)(self.h, dy.vp, dx.vp))
        return dy.host()

    def dinv(self):
        d = np.zeros(self.n)
        L.check(LIB().fvh_precond_dinv(self.h, L.dptr(d)))
        return d


def _inputs(nx, ny):
    mesh = F.channel(nx, ny)
    dm = mesh.device()
    rp, ci = dm.pattern()
    rng = np.random.default_rng(nx + 1000 * ny)
    rows = np.repeat(np.arange(mesh.ncells), np.diff(rp))
    mats = [np.where(rows == ci, -4.2 - rng.random(ci.size), 0.7 + 0.5 * rng.random(ci.size)) for _ in range(2)]
    return mesh, dm, mats, rng.standard_normal(mesh.ncells), rows == ci


SIZES = [(7, 1), (1, 7), (20, 12), (65, 65), (130, 70)]


@pytest.mark.parametrize("nx,ny", SIZES)
@pytest.mark.parametrize("kind", [L.PRECOND_DILU, L.PRECOND_ILU0])
def test_an_update_forgets_a_singular_matrix(kind, nx, ny):
    """No entries, a zero pivot and a NaN, each followed by a regular matrix:
    the applies are those of a fresh equation."""
    mesh, dm, (A, _), x, on_diag = _inputs(nx, ny)
    n = mesh.ncells
    with _Eq(dm, n) as fresh, _Eq(dm, n) as used:
        for eq in (fresh, used):
            eq.set(kind)
        fresh.update(A)
        want = fresh.apply(x), fresh.apply(x, True)
        assert np.isfinite(want[0]).all() and np.isfinite(want[1]).all()
        zero, nan = A.copy(), A.copy()
        zero[np.nonzero(on_diag)[0][n // 2]] = 0.0
        nan[np.nonzero(on_diag)[0][n - 1]] = np.nan
        for bad in (np.zeros_like(A), zero, nan):
            used.update(bad)
            used.apply(x), used.apply(x, True)
            used.update(A)
            assert same_bits(used.apply(x), want[0]), (kind, nx, ny)
            assert same_bits(used.apply(x, True), want[1]), (kind, nx, ny)


@pytest.mark.parametrize("nx,ny", SIZES)
def test_dilu_and_ilu0_in_turn_on_one_equation(nx, ny):
    """Each applies its own last update, DILU's reciprocal diagonal included;
    one that was never updated refuses, in either precision."""
    mesh, dm, (A, B), x, _ = _inputs(nx, ny)
    n = mesh.ncells
    want = {}
    for kind, M in ((L.PRECOND_DILU, A), (L.PRECOND_ILU0, B)):
        with _Eq(dm, n) as eq:
            eq.set(kind)
            eq.update(M)
            want[kind] = eq.apply(x), eq.apply(x, True), eq.dinv() if kind == L.PRECOND_DILU else None
    for first, second in ((L.PRECOND_DILU, L.PRECOND_ILU0), (L.PRECOND_ILU0, L.PRECOND_DILU)):
        mats = {L.PRECOND_DILU: A, L.PRECOND_ILU0: B}
        with _Eq(dm, n) as eq:
            eq.set(first)
            eq.update(mats[first])
            eq.set(second)
            dx, dy = L.DeviceArray.from_host(x), L.DeviceArray(n)
            fx, fy = L.DeviceArray.from_host(x.astype(np.float32)), L.DeviceArray(n, np.float32)
            if min(nx, ny) > 1:  # on the band sweeps (a single row of cells is on the level walk)
                assert LIB().fvh_precond_apply(eq.h, dy.vp, dx.vp) == L.FVH_ERR_ARG
                assert LIB().fvh_precond_apply_f32(eq.h, fy.vp, fx.vp) == L.FVH_ERR_ARG
            eq.update(mats[second])
            assert same_bits(eq.apply(x), want[second][0]) and same_bits(eq.apply(x, True), want[second][1])
            if second == L.PRECOND_DILU:
                assert same_bits(eq.dinv(), want[L.PRECOND_DILU][2])
            if min(nx, ny) > 1:  # as updated before (elsewhere a set-up allocates anew)
                eq.set(first)
                assert same_bits(eq.apply(x), want[first][0]) and same_bits(eq.apply(x, True), want[first][1])
                eq.set(L.PRECOND_DILU)
                assert same_bits(eq.dinv(), want[L.PRECOND_DILU][2])
