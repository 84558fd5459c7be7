"""The one-point-per-thread stencil step (complex blocks, non-orthogonal cells,
and real orthogonal ones without the run-vector kernel) at the edges of its launch shapes, against the oracle: rows shorter
than two ghost widths (both copies of a point), fewer than 12 planes (no march
once around z) and z-chunks, rows at the limits of each LDS pitch, a band of
one row, grids smaller than a workgroup.  H applies and a filter (the
Y_(k-2) stream) of every element type that takes the path, alone and in a
batch.  Bars of the other stencil tests: 1e-12 (FP64) and 2e-6 (single
precision) per apply, 1e-11 and 2e-5 per filter."""
import numpy as np
import pytest

from systems import FCC_PRIMITIVE, System

pytestmark = pytest.mark.gpu
SI2 = np.array([[0.05, 0.1, 0.2], [0.5, 0.55, 0.45]])
DTYPES = [np.float64, np.complex128, np.float32, np.complex64]
GRIDS = [(6, 6, 6), (7, 9, 11), (11, 8, 12), (12, 6, 13), (28, 7, 9), (29, 13, 8), (52, 6, 14), (53, 9, 7),
         (64, 6, 13), (65, 9, 7), (116, 7, 12), (23, 37, 13)]


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


def system(n, skew):
    # an uneven spacing along x, y and z, so that no two axes are alike
    L = np.array(n) * np.array([0.5, 0.55, 0.6])
    if skew:
        s = System(n, 1.0, SI2, latvec=FCC_PRIMITIVE * np.sqrt(2.0) * L[:, None], with_nonlocal=False)
    else:
        s = System(n, L, SI2, with_nonlocal=False)
    lens = np.sqrt((s.latvec ** 2).sum(axis=1))
    s.kpt = tuple(2 * np.pi * np.array([0.21, -0.13, 0.34]) / lens)
    return s


@pytest.mark.parametrize("n", GRIDS)
@pytest.mark.parametrize("skew", [False, True])
def test_points_step_matches_oracle(n, skew):
    from lynx_amd import _lib as L, core
    s = system(n, skew)
    op, H = s.oracle_op(), s.hamiltonian()
    lo, hi = s.veff.min() - 0.5, 80.0
    lc = lo + 0.3 * (hi - lo)
    for dt in DTYPES:
        cplx = np.dtype(dt).kind == "c"
        single = np.dtype(dt).itemsize == (8 if cplx else 4)
        k = s.kpt if cplx else (0.0, 0.0, 0.0)
        op.set_kpoint(k)
        H.set_kpoint(k)
        X = s.random_block(3, 41, cplx).astype(dt)
        ref = op.apply(X.astype(complex if cplx else float), s.veff, c=-0.2)
        for shape in [(t, d, z) for t in (256, 512) for d in (1, 2) for z in (1, 2, (n[2] + 2) // 3)]:
            L.check(L.lib().lynx_set_stencil_config(H.ctx, *shape, 0), H.ctx)
            got = H._apply(X.T.copy(), s.veff, -0.2, dt).reshape(3, -1).T
            assert rel(got, ref) < (2e-6 if single else 1e-12), (dt, shape)
        L.check(L.lib().lynx_set_stencil_config(H.ctx, 0, 0, 0, 0), H.ctx)
        ref = op.cheb_filter(X.astype(complex if cplx else float), s.veff, lc, lo, hi, 5)
        bf = core.BatchFilter([(H, k), (H, k)])
        got = bf.filter([X, X[:, :2]], 5, lc, lo, hi, dtype=dt)
        assert rel(got[0], ref) < (2e-5 if single else 1e-11), dt
        assert rel(got[1], ref[:, :2]) < (2e-5 if single else 1e-11), dt
        bf.close()
        Y = np.zeros_like(X, order="F")
        Xf = np.asfortranarray(X)
        L.check(L.lib().lynx_cheb_filter(H.ctx, L.dtype_code(dt), L.vptr(Xf), s.nd, L.vptr(Y), s.nd, 3, 5, lc, lo, hi,
                                         L.MEM_HOST), H.ctx)
        assert rel(Y, ref) < (2e-5 if single else 1e-11), dt


@pytest.mark.parametrize("n", [(60, 9, 14), (40, 18, 12), (72, 11, 13), (116, 6, 13)])
@pytest.mark.parametrize("skew", [False, True])
def test_batch_shapes_match_oracle(n, skew):
    # rows whose LDS leaves few waves on a CU: marches beyond the z boundary
    # instead of around it, and complex128 rows of more than three halo points
    # per thread in fewer threads
    from lynx_amd import core
    s = system(n, skew)
    op, H = s.oracle_op(), s.hamiltonian()
    H.set_veff(s.veff)
    lo, hi = s.veff.min() - 0.5, 80.0
    lc = lo + 0.3 * (hi - lo)
    for dt in DTYPES:
        cplx = np.dtype(dt).kind == "c"
        single = np.dtype(dt).itemsize == (8 if cplx else 4)
        k = s.kpt if cplx else (0.0, 0.0, 0.0)
        op.set_kpoint(k)
        X = s.random_block(3, 43, cplx).astype(dt)
        ref = op.cheb_filter(X.astype(complex if cplx else float), s.veff, lc, lo, hi, 4)
        bf = core.BatchFilter([(H, k), (H, k)])
        got = bf.filter([X, X[:, :1]], 4, lc, lo, hi, dtype=dt)
        assert rel(got[0], ref) < (2e-5 if single else 1e-11), dt
        assert rel(got[1], ref[:, :1]) < (2e-5 if single else 1e-11), dt
        bf.close()
