"""The LDL block solves (inverted triangles per range) at the sizes where their
cases meet: ranges of 64, 65, 80 and 81 rows (one or two row groups, one range
or a split), separators longer than one block's 64 rows, rows longer than the
entries a wave loads at once, and separators cut at 512 rows.  Against the
row-by-row substitution on the same matrix.  Both solve A z = x backward
stably, so each residual is a small multiple of n^(1/2) eps cond-free: 1e-13
covers the measured 2e-15 with the growth of a separator's inverse (its
entries are bounded by 1 for these M-matrices)."""
import ctypes as C

import numpy as np
import pytest

import fvmhip as F
from fvmhip import _lib as L

pytestmark = pytest.mark.gpu
LIB = L.lib


def _apply(dm, vals, x, monkeypatch, blocks):
    monkeypatch.setenv("FVH_LDL_RANGES", "1" if blocks else "0")
    eq, nz = C.c_void_p(), C.c_void_p()
    L.check(LIB().fvh_eqn_create(dm.h, C.byref(eq)))
    try:
        L.check(LIB().fvh_eqn_arrays(eq, C.byref(nz), None))
        L.check(LIB().fvh_memcpy(nz, vals.ctypes.data_as(C.c_void_p), vals.nbytes))
        L.check(LIB().fvh_precond_set(eq, L.PRECOND_LDL, None))
        L.check(LIB().fvh_precond_update(eq))
        dx, dy, dr = L.DeviceArray.from_host(x), L.DeviceArray(x.size), L.DeviceArray(x.size)
        L.check(LIB().fvh_precond_apply(eq, dy.vp, dx.vp), "fvh_precond_apply")
        L.check(LIB().fvh_spmv(eq, dy.vp, dr.vp))
        y = dy.host()
        return y, np.linalg.norm(dr.host() - x) / np.linalg.norm(x)
    finally:
        LIB().fvh_eqn_destroy(eq)


@pytest.mark.parametrize("nx,ny", [(2, 1), (8, 8), (13, 5), (8, 10), (9, 9), (1, 300), (70, 66), (310, 140), (530, 520)])
def test_block_solves_against_substitution(nx, ny, monkeypatch):
    mesh = F.channel(nx, ny)
    dm = mesh.device()
    rp, ci = dm.pattern()
    rows = np.repeat(np.arange(mesh.ncells), np.diff(rp))
    # symmetric: the entry of a pair depends on the pair alone
    pair = np.minimum(rows, ci) * 7 + np.maximum(rows, ci)
    vals = np.where(rows == ci, 4.05, -0.9 - 0.1 * np.sin(pair * 0.37))
    x = np.random.default_rng(nx).standard_normal(mesh.ncells)
    got, res = _apply(dm, vals, x, monkeypatch, True)
    want, res0 = _apply(dm, vals, x, monkeypatch, False)
    diff = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"{nx}x{ny}: residual {res:.1e} (substitution {res0:.1e}), difference {diff:.1e}", flush=True)
    # the difference is the residuals' times the condition number (<= 8.05 / 0.05)
    assert res <= 1e-13 and diff <= 1e-11


@pytest.mark.parametrize("nx,ny", [(13, 5), (70, 66), (310, 140)])
@pytest.mark.parametrize("shift", [0.5, 1.3, 2.7])
def test_indefinite_matrices(nx, ny, shift, monkeypatch):
    """Ranges cut where their inverse grows (down to single rows): the residual
    is the substitution's.  Two solves of like accuracy differ by a factor of
    about e^0.6 either way; 8 is more than three of that (uncut, 310 x 140 and
    1.3: 11 times the substitution's)."""
    mesh = F.channel(nx, ny)
    dm = mesh.device()
    rp, ci = dm.pattern()
    rows = np.repeat(np.arange(mesh.ncells), np.diff(rp))
    vals = np.where(rows == ci, 4.0 - shift, -1.0)
    x = np.random.default_rng(nx).standard_normal(mesh.ncells)
    got, res = _apply(dm, vals, x, monkeypatch, True)
    want, res0 = _apply(dm, vals, x, monkeypatch, False)
    print(f"{nx}x{ny} {shift}: residual {res:.1e} (substitution {res0:.1e})", flush=True)
    assert res <= 8 * res0
