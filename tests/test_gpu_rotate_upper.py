"""Cholesky-QR of wide real FP64 blocks through lynx_orthogonalize: the Gram
tiles of 96 columns and the in-place triangular rotation in blocks of 48 and
strips of 192 columns, against numpy.  Widths at those edges and beyond the
narrow kernels' 64; grids whose points fill no workgroup of 64 and no 16-row
step, with an odd and an even leading dimension.

Tolerance: a random block of n <= 400 of 1287 or more columns has kappa(X) <
4; Gram, Cholesky inverse and product each round to about n 2^-53 kappa^2 =
7e-13 of the result's norm (1e-11 asserted)."""
import numpy as np
import pytest

from systems import A_SI, DIAMOND, System

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid,pad", [((11, 9, 13), 0), ((11, 9, 13), 1), ((12, 12, 13), 2)])
def test_wide_cholesky_qr_matches_numpy(grid, pad):
    from lynx_amd import _lib as L
    s = System(grid, A_SI, DIAMOND)
    H = s.hamiltonian()
    dv = abs(np.linalg.det(s.latvec)) / s.nd
    ld = s.nd + pad
    for n in (65, 79, 80, 95, 96, 97, 144, 145, 191, 192, 193, 240, 257, 400):
        X = np.full((ld, n), np.nan, order="F")     # padding rows are not touched
        X[:s.nd] = s.random_block(n, 7 + n, False)
        x = X[:s.nd].copy()
        L.check(L.lib().lynx_orthogonalize(H.ctx, L.F64, L.vptr(X), ld, n, L.MEM_HOST), H.ctx)
        r = np.linalg.cholesky(dv * x.T @ x).T
        ref = np.linalg.solve(r.T, x.T).T
        assert np.linalg.norm(X[:s.nd] - ref) < 1e-11 * np.linalg.norm(ref), n
        assert np.isnan(X[s.nd:]).all(), n
