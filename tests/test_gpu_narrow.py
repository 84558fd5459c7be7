"""Narrow blocks (up to 64 real or 32 complex columns) on the dense kernels:
the Gram product, the Cholesky-QR, the projection and the eigensolve of
lynx_chefsi_solve, against numpy in double precision.  Widths at the edges of
the 16-column tiles and of the covered range (one more column takes the
general path); an odd number of rows (columns off the 16-byte boundary, a
partial 16-row step) and a padded leading dimension.

Tolerances: a sum of 1287 or 1728 products of random signs and values below
one rounds to about 1e-14 of the largest Gram entry (1e-12 asserted); the
random block's condition number is below 1e3, so one Cholesky-QR leaves
orthonormality to about kappa^2 * 1e-16 (1e-9 asserted); the eigensolve is
backward stable, n * 2^-53 of the norm (1e-11 of the largest Ritz value
asserted)."""
import ctypes

import numpy as np
import pytest

from systems import A_SI, DIAMOND, System

pytestmark = pytest.mark.gpu
KPT = (0.11, 0.23, -0.07)


@pytest.fixture(scope="module")
def hams():
    out = {}
    for n in ((11, 9, 13), (12, 12, 12)):
        s = System(n, A_SI, DIAMOND, kpt=KPT)
        H = s.hamiltonian()
        H.set_veff(s.veff)
        out[n] = (s, H, abs(np.linalg.det(s.latvec)) / s.nd)
    return out


CASES = [((11, 9, 13), n, False) for n in (1, 15, 16, 17, 32, 33, 48, 63, 64, 65)]
CASES += [((12, 12, 12), n, False) for n in (24, 49)]
CASES += [((11, 9, 13), n, True) for n in (1, 12, 16, 17, 32, 33)] + [((12, 12, 12), 12, True)]


@pytest.mark.parametrize("grid,n,cplx", CASES)
def test_narrow_blocks_match_numpy(hams, grid, n, cplx):
    from lynx_amd import _lib as L
    s, H, dv = hams[grid]
    lib, ctx = L.lib(), H.ctx
    code = L.C128 if cplx else L.F64
    ld = s.nd + 3                                   # a padded leading dimension
    X = np.zeros((ld, n), complex if cplx else float, order="F")
    X[:s.nd] = s.random_block(n, 5 + n, cplx)
    x = X[:s.nd].copy()
    S = np.zeros((n, n), X.dtype, order="F")
    L.check(lib.lynx_gram(ctx, code, L.vptr(X), ld, L.vptr(X), ld, n, L.vptr(S), L.MEM_HOST), ctx)
    ref = dv * x.conj().T @ x
    assert np.abs(S - ref).max() < 1e-12 * np.abs(ref).max()

    # Cholesky-QR: X R^-1 with R^H R = S
    L.check(lib.lynx_orthogonalize(ctx, code, L.vptr(X), ld, n, L.MEM_HOST), ctx)
    q = X[:s.nd]
    assert np.abs(dv * q.conj().T @ q - np.eye(n)).max() < 1e-9
    r = np.linalg.cholesky(ref).conj().T
    assert np.abs(q @ r - x).max() < 1e-11 * np.abs(x).max() * n

    # one pass: orthonormal Ritz vectors that diagonalise the projection
    lo, hi = s.veff.min() - 1.0, 80.0
    P = np.zeros((ld, n), X.dtype, order="F")
    P[:s.nd] = x
    eig = np.zeros(n)
    lc = ctypes.c_double()
    L.check(lib.lynx_chefsi_solve(ctx, code, L.vptr(P), ld, n, L.dptr(eig), lo + 0.4 * (hi - lo), lo, hi, 2,
                                  ctypes.byref(lc), L.MEM_HOST), ctx)
    p = P[:s.nd]
    assert np.all(np.diff(eig) >= 0) and lc.value == eig[-1] + 0.1
    assert np.abs(dv * p.conj().T @ p - np.eye(n)).max() < 1e-9
    T = np.zeros((n, n), X.dtype, order="F")
    L.check(lib.lynx_project_hamiltonian(ctx, code, L.vptr(P), ld, n, L.vptr(T), L.MEM_HOST), ctx)
    assert np.abs(T - T.conj().T).max() == 0.0
    assert np.abs(T - np.diag(eig)).max() < 1e-9 * np.abs(eig).max()
    assert np.all(P[s.nd:] == 0)


@pytest.mark.parametrize("cplx", [False, True])
def test_dependent_columns_are_refused(hams, cplx):
    """A zero column has no Cholesky factor: the status names it and the
    block is left as it was."""
    from lynx_amd import _lib as L
    s, H, _ = hams[(12, 12, 12)]
    X = s.random_block(12, 3, cplx)
    X[:, 7] = 0.0
    keep = X.copy()
    st = L.lib().lynx_orthogonalize(H.ctx, L.C128 if cplx else L.F64, L.vptr(X), s.nd, 12, L.MEM_HOST)
    assert st == L.E_CHOLESKY
    assert np.array_equal(X, keep)
