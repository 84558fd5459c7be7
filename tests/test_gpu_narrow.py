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


def narrow_eig(mats):
    """The library's kernel for narrow_eig on a stack of equal matrices:
    (vectors, eigenvalues, info), of buffers that held 7 before the call."""
    from lynx_amd import _lib as L
    from lynx_amd.hipmem import DeviceArray, synchronize
    units, n = mats.shape[:2]
    f = L.lib()._ZN4lynx3gpu10narrow_eigEiPviiPdPiP12ihipStream_t
    f.restype = None
    f.argtypes = [ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p,
                  ctypes.c_void_p]
    M = np.ascontiguousarray(mats.transpose(0, 2, 1))
    ev, info = np.full((units, n), 7.0), np.full(units, 7, np.int32)
    d = [DeviceArray.from_numpy(a) for a in (M, ev, info)]
    f(L.C128 if np.iscomplexobj(M) else L.F64, d[0].ptr, n, units, d[1].ptr, d[2].ptr, None)
    synchronize()
    for a, b in zip((M, ev, info), d):
        b.download(a)
        b.free()
    return M.transpose(0, 2, 1), ev, info


def hermitian(n, cplx, seed):
    rng = np.random.default_rng(seed)
    a = rng.normal(size=(n, n)) + (1j * rng.normal(size=(n, n)) if cplx else 0.0)
    return a + a.conj().T


@pytest.mark.parametrize("n,cplx", [(1, False), (24, False), (33, False), (64, False), (1, True), (12, True),
                                    (32, True)])
def test_eigensolve_refuses_values_that_are_not_finite(hams, n, cplx):
    # one bad value anywhere in the upper triangle: that matrix is refused and
    # left alone with its eigenvalues, its neighbours are solved
    good = hermitian(n, cplx, 3)
    ref = np.linalg.eigvalsh(good)
    for bad in (np.nan, np.inf, -np.inf) + ((1j * np.inf, complex(0.0, np.nan)) if cplx and n > 1 else ()):
        for at in {(0, 0), (n - 1, n - 1), (0, n - 1), (n // 2, n - 1)}:
            if np.iscomplex(bad) and at[0] == at[1]:
                continue                        # a diagonal's imaginary part is not read
            mats = np.stack([good, good, good])
            mats[1][at] = bad
            keep = mats[1].copy()
            v, ev, info = narrow_eig(mats)
            assert list(info) == [0, 1, 0], (bad, at)
            assert np.array_equal(v[1], keep, equal_nan=True) and np.all(ev[1] == 7.0)
            for u in (0, 2):
                assert np.abs(ev[u] - ref).max() < 1e-13 * n * np.abs(ref).max()


@pytest.mark.parametrize("n,cplx", [(1, False), (24, False), (64, False), (12, True), (32, True)])
def test_eigensolve_scales_with_its_matrix(hams, n, cplx):
    # entries whose squares overflow or vanish: a power of two changes the
    # eigenvalues by that power and the vectors not at all
    a = hermitian(n, cplx, 5)
    v, ev, info = narrow_eig(np.stack([np.ldexp(a.view(float), k).view(a.dtype) for k in (0, 600, 1000, -600, -900)]))
    assert np.all(info == 0)
    assert np.abs(a @ v[0] - v[0] * ev[0]).max() < 1e-13 * n * np.abs(ev[0]).max()
    for i, k in enumerate((0, 600, 1000, -600, -900)):
        assert np.array_equal(ev[i], np.ldexp(ev[0], k)) and np.array_equal(v[i], v[0]), k
    v, ev, info = narrow_eig(np.zeros_like(a)[None])
    assert info[0] == 0 and np.all(ev == 0.0) and np.array_equal(v[0], np.eye(n))
