"""The run-vector stencil kernels with two runs per thread (adjacent rows that
share their LDS reads) at the edges of the bands, against the oracle: an odd
number of rows (the last thread row owns one run and needs the row beyond the
band, wrapped or not), one row, fewer rows than threads, several bands, runs
of two and of four points, both directions of a
z-chunk, chunks of three planes.  Bars of the other
stencil tests: 1e-12 (FP64) and 2e-6 (single precision) per apply, 1e-11 and
2e-5 per filter."""
import numpy as np
import pytest

from systems import System

pytestmark = pytest.mark.gpu
SI2 = np.array([[0.05, 0.1, 0.2], [0.5, 0.55, 0.45]])
GRIDS = [(12, 6, 13), (14, 7, 12), (16, 9, 6), (28, 17, 9), (30, 33, 14), (60, 15, 8), (90, 11, 7), (104, 23, 8),
         (116, 7, 8)]


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


@pytest.mark.parametrize("n", GRIDS)
def test_run_vector_rows_match_oracle(n):
    from lynx_amd import _lib as L
    s = System(n, np.array(n) * np.array([0.5, 0.55, 0.6]), SI2, with_nonlocal=False)
    op, H = s.oracle_op(), s.hamiltonian()
    lo, hi = s.veff.min() - 0.5, 80.0
    lc = lo + 0.3 * (hi - lo)
    for dt in (np.float64, np.float32):
        single = dt is np.float32
        X = s.random_block(3, 43, False).astype(dt)
        one = op.apply(X.astype(float), s.veff, c=-0.2)
        five = op.cheb_filter(X.astype(float), s.veff, lc, lo, hi, 5)
        for shape in [(t, d, z, v) for t in (256, 512) for d in (1, 2) for z in (1, 2, (n[2] + 2) // 3) for v in (1, 2, 3, 5, 6, 7)]:
            L.check(L.lib().lynx_set_stencil_config(H.ctx, *shape), H.ctx)
            got = H._apply(X.T.copy(), s.veff, -0.2, dt).reshape(3, -1).T
            assert rel(got, one) < (2e-6 if single else 1e-12), (dt, shape)
            Y = np.zeros_like(X, order="F")
            Xf = np.asfortranarray(X)
            L.check(L.lib().lynx_cheb_filter(H.ctx, L.dtype_code(dt), L.vptr(Xf), s.nd, L.vptr(Y), s.nd, 3, 5, lc, lo,
                                             hi, L.MEM_HOST), H.ctx)
            assert rel(Y, five) < (2e-5 if single else 1e-11), (dt, shape)
        L.check(L.lib().lynx_set_stencil_config(H.ctx, 0, 0, 0, 0), H.ctx)
