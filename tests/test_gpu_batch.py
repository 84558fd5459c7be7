"""Batched filter (lynx_batch_*): many units in one launch per kernel per
Chebyshev step, replayed from a HIP graph.  Every unit's result is checked
against the oracle's filter of that unit alone (FP64 1e-11, FP32 2e-5), and
graph replays against eager launches of the same plan (bitwise)."""
import ctypes

import numpy as np
import pytest

import oracle
from systems import A_SI, DIAMOND, System, displace, si2_fcc, si8

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / max(np.linalg.norm(np.asarray(b)), 1e-300))


def kvec(s, red):
    L = np.sqrt((s.latvec ** 2).sum(axis=1))
    return tuple(2 * np.pi * np.asarray(red) / L)


def _bounds(i):
    return 0.3 + 0.05 * i, -0.6 - 0.02 * i, 60.0 + 3.0 * i


@pytest.fixture(scope="module")
def fcc_kbatch():
    # k-points of one FCC Si2 cell sharing one Hamiltonian
    from lynx_amd import core
    s = si2_fcc(16)
    H = s.hamiltonian()
    H.set_veff(s.veff)
    reds = [(0.0, 0.0, 0.0), (0.25, 0.0, 0.0), (0.25, 0.25, 0.0), (0.5, 0.25, -0.25), (-0.125, 0.375, 0.5)]
    ks = [kvec(s, r) for r in reds]
    return s, H, ks, core


@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-11), (np.complex64, 2e-5)])
def test_kpoint_batch_matches_per_kpoint_oracle(fcc_kbatch, dtype, tol):
    s, H, ks, core = fcc_kbatch
    bf = core.BatchFilter([(H, k) for k in ks])
    blocks = [s.random_block(3 + (i % 2), 50 + i, complex_=True) for i in range(len(ks))]
    deg = 8
    lc, lo, hi = zip(*[_bounds(i) for i in range(len(ks))])
    got = bf.filter(blocks, deg, lc, lo, hi, dtype=dtype)
    op = s.oracle_op()
    for i, k in enumerate(ks):
        op.set_kpoint(k)
        ref = op.cheb_filter(blocks[i], s.veff, lc[i], lo[i], hi[i], deg)
        assert rel(got[i], ref) < tol, (i, k)
    bf.close()


@pytest.mark.parametrize("dtype,tol", [(np.float64, 1e-11), (np.float32, 2e-5)])
def test_heterogeneous_batch_matches_oracle(dtype, tol):
    # orthogonal and non-orthogonal cells, different grids and band counts,
    # one without projectors; rows of 20 points (16-byte float runs) and of
    # 26 (8-byte float runs)
    from lynx_amd import core
    systems = [si8(20), si2_fcc(18), System((20, 22, 24), A_SI, displace(DIAMOND, A_SI, 0.05, seed=4)),
               si8(16, with_nonlocal=False), System((26, 20, 22), A_SI, displace(DIAMOND, A_SI, 0.05, seed=5))]
    Hs = []
    for s in systems:
        H = s.hamiltonian()
        H.set_veff(s.veff)
        Hs.append(H)
    bf = core.BatchFilter([(H, None) for H in Hs])
    blocks = [s.random_block(2 + i, 60 + i) for i, s in enumerate(systems)]
    deg = 7
    lc, lo, hi = zip(*[_bounds(i) for i in range(len(systems))])
    got = bf.filter(blocks, deg, lc, lo, hi, dtype=dtype)
    for i, s in enumerate(systems):
        ref = s.oracle_op().cheb_filter(blocks[i], s.veff, lc[i], lo[i], hi[i], deg)
        assert rel(got[i], ref) < tol, i
    bf.close()


@pytest.mark.parametrize("dtype,tol", [(np.complex128, 1e-11), (np.complex64, 2e-5), (np.float64, 1e-11),
                                       (np.float32, 2e-5)])
def test_batch_gather_by_parts(dtype, tol):
    # atoms with more than 1024 sphere points (BaTiO3 at 20^3: the La
    # stand-in has 1955 over its images, Zr 1221) are gathered by parts of
    # 256 points and 8 columns, then the parts are summed per atom; 3 and 11
    # columns (a partial column group), two k-points or Gamma twice
    from lynx_amd import core
    from systems import batio3
    s = batio3(0, n=20)
    H = s.hamiltonian()
    H.set_veff(s.veff)
    cplx = np.dtype(dtype).kind == "c"
    ks = [kvec(s, (0.25, -0.125, 0.375)), kvec(s, (0.0, 0.5, 0.25))] if cplx else [None, None]
    bf = core.BatchFilter([(H, k) for k in ks])
    blocks = [s.random_block(3, 120, complex_=cplx), s.random_block(11, 121, complex_=cplx)]
    deg = 6
    lc, lo, hi = zip(*[_bounds(i) for i in range(2)])
    got = bf.filter(blocks, deg, lc, lo, hi, dtype=dtype)
    op = s.oracle_op()
    for i, k in enumerate(ks):
        op.set_kpoint(k if k is not None else (0.0, 0.0, 0.0))
        ref = op.cheb_filter(blocks[i], s.veff, lc[i], lo[i], hi[i], deg)
        assert rel(got[i], ref) < tol, (i, k)
    bf.close()


def test_graph_replays_match_eager_launches(fcc_kbatch):
    # the same plan run eagerly and from the captured graph, several calls
    # in a row with different inputs and bounds and other GPU work between
    s, H, ks, core = fcc_kbatch
    units = [(H, k) for k in ks[:3]]
    g = core.BatchFilter(units, graph=True)
    e = core.BatchFilter(units, graph=False)
    for rep in range(3):
        blocks = [s.random_block(4, 70 + 10 * rep + i, complex_=True) for i in range(3)]
        lc, lo, hi = zip(*[_bounds(i + rep) for i in range(3)])
        yg = g.filter(blocks, 9, lc, lo, hi, dtype=np.complex128)
        H.apply_kpt(H.halo, blocks[0].T.copy(), s.veff, ks[1])      # unrelated work on the context's stream
        ye = e.filter(blocks, 9, lc, lo, hi, dtype=np.complex128)
        for a, b in zip(yg, ye):
            assert np.array_equal(a, b), rep
    ms, launches = g.last_timing()
    # nine stencil steps; the spheres share no grid point, so the scatter of a
    # step and the gather of the next are one launch
    assert launches == 9 + (9 + 1) and ms > 0
    g.close()
    e.close()


@pytest.mark.parametrize("sizes,disjoint,per_step,more", [((), True, 1, 0), ((16, 33), True, 2, 1),
                                                          ((16, 33), False, 3, 0), ((1025, 40), True, 4, 0)])
def test_launch_counts(sizes, disjoint, per_step, more):
    # without projectors; scatter and next gather in one launch; apart (a grid
    # point in two spheres); apart, with a gather by parts (large spheres).
    # Alone the gather of large spheres is one launch
    from lynx_amd import _lib as L, core
    from test_gpu_nonlocal import N, raw_projectors
    s = System(N, np.array([6.0, 5.8, 5.5]), np.array([[0.3, 0.4, 0.5]]), with_nonlocal=False)
    H = s.hamiltonian()
    if sizes:
        lat, grid, st, dom, halo = s.core
        raw = raw_projectors(5, sizes, disjoint, 7, np.sqrt((s.latvec ** 2).sum(axis=1)))[0]
        H = core.Hamiltonian(0).setup(st, dom, grid, halo, core.NonlocalProjector().setup_raw(**raw))
    H.set_veff(s.veff)
    lc, lo, hi = _bounds(0)
    X = s.random_block(3, 5)
    for graph in (True, False):
        bf = core.BatchFilter([(H, None)], graph=graph)
        for degree in (1, 2, 7):
            bf.filter([X], degree, lc, lo, hi)
            assert bf.last_timing()[1] == per_step * degree + more, (graph, degree)
        bf.close()
    L.check(L.lib().lynx_set_timing(H.ctx, 1), H.ctx)
    Y = np.zeros_like(X, order="F")
    L.check(L.lib().lynx_cheb_filter(H.ctx, L.F64, L.vptr(X), s.nd, L.vptr(Y), s.nd, 3, 7, lc, lo, hi, L.MEM_HOST),
            H.ctx)
    ms, n = (ctypes.c_double * 4)(), (ctypes.c_int * 4)()
    L.check(L.lib().lynx_last_filter_timing(H.ctx, ms, n), H.ctx)
    assert list(n)[1:] == ([7, 0, 0] if not sizes else [7, 1, 7] if more else [7, 7, 7])


def test_batch_errors():
    from lynx_amd import core, _lib as L
    s = si8(16)
    H = s.hamiltonian()
    H.set_veff(s.veff)
    bf = core.BatchFilter([(H, None)])
    with pytest.raises(L.LynxError):
        bf.filter([s.random_block(2, 1)], 5, [50.0], [-1.0], [40.0])   # eig_max below lambda_cutoff
    bf.close()


def test_batch_follows_a_reconfigured_context():
    # a member context set up again after the batch was made (other atoms on
    # the same grid, then a larger grid): the batch rebuilds its plan, phase
    # tables and graph and matches the oracle of the new set-up
    from lynx_amd import core as C
    s1 = System(18, A_SI, displace(DIAMOND, A_SI, 0.05, seed=21))
    H = s1.hamiltonian()
    H.set_veff(s1.veff)
    k = kvec(s1, (0.25, -0.125, 0.0))
    bf = C.BatchFilter([(H, k), (H, None)])
    lc, lo, hi = zip(*[_bounds(i) for i in range(2)])
    systems = (s1, System(18, A_SI, displace(DIAMOND, A_SI, 0.08, seed=22)),
               System(20, A_SI, displace(DIAMOND, A_SI, 0.05, seed=23)))
    for rep, s in enumerate(systems):
        if rep > 0:
            lat = C.Lattice(s.latvec, C.CellType.Orthogonal)
            grid = C.FDGrid(*s.n, lat)
            st = C.FDStencil(12, grid, lat)
            dom = C.Domain(grid)
            vnl = C.NonlocalProjector().setup_atoms(s.psp_files, s.types, s.frac, True)
            H.setup(st, dom, grid, C.HaloExchange(dom, st.FDn()), vnl)
            H.set_veff(s.veff)
        blocks = [s.random_block(3, 90 + rep, complex_=True), s.random_block(2, 95 + rep, complex_=True)]
        op = s.oracle_op()
        for graph_pass in range(2):
            got = bf.filter(blocks, 6, lc, lo, hi, dtype=np.complex128)
            for i, kk in enumerate((k, (0.0, 0.0, 0.0))):
                op.set_kpoint(kk)
                ref = op.cheb_filter(blocks[i], s.veff, lc[i], lo[i], hi[i], 6)
                assert rel(got[i], ref) < 1e-11, (rep, graph_pass, i)
    bf.close()
