"""Nonlocal projector kernels at the edges of their tiles: atoms of 1, 16, 17,
33 and 1025 sphere points (tiles hold 16; over 1024 the atom takes the
gather of large spheres), 5, 16 and 20 projectors (padded to 8, 16 and 32),
column counts around the groups of 16 real or 8 complex columns, several
images per atom with Bloch phases, spheres that share no grid point (the
scatter and the next step's gather are one launch) and spheres that do.

Random projectors through lynx_set_nonlocal.  The reference is the oracle's
local operator plus a dense V_nl in numpy: one H apply and a degree-4 filter,
alone and in a batch.  Sums of up to 1025 products: 1e-12 (FP64) and 5e-6
(single precision) relative per apply, 1e-11 and 5e-5 per filter; bfloat16
storage 2^-8 per value and step, 2e-2."""
import numpy as np
import pytest

from systems import System

pytestmark = pytest.mark.gpu
N = (14, 13, 12)
DEG = 4


def raw_projectors(nproj, sizes, disjoint, seed, L):
    """Atoms with the given numbers of points, each split over two images;
    scaled so that V_nl stays of order one."""
    rng = np.random.default_rng(seed)
    nd = int(np.prod(N))
    perm = rng.permutation(nd)
    img, gpos, chi, shift, displ, gamma = [], [], [], [], [0], []
    used = 0
    for a, n in enumerate(sizes):
        pts = perm[used:used + n] if disjoint else rng.choice(nd // 2, n, replace=False)
        used += n
        np_a = max(1, nproj - a)
        for part in (pts[:n // 3], pts[n // 3:]):
            if len(part) == 0:
                continue
            img.append((a, len(part), np_a))
            gpos.append(part)
            chi.append(rng.normal(size=(len(part), np_a)))
            shift.append(rng.integers(-1, 2, 3) * L)
        displ.append(displ[-1] + np_a)
        gamma.append(rng.uniform(-1.0, 1.0, np_a) / n)
    return dict(img_atom=[i[0] for i in img], img_ndc=[i[1] for i in img], img_nproj=[i[2] for i in img],
                gpos=np.concatenate(gpos), chi=np.concatenate([c.ravel(order="F") for c in chi]),
                img_shift=np.concatenate(shift), n_atom=len(sizes), ip_displ=displ, gamma=np.concatenate(gamma)), \
        list(zip([i[0] for i in img], gpos, chi, shift)), displ, np.concatenate(gamma)


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - np.asarray(b)) / np.linalg.norm(np.asarray(b)))


def bf16_round(x):
    u = np.asarray(x, np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) >> 16).astype(np.uint16)


SIZES = [(1, 16, 17, 33), (1025, 40)]


@pytest.mark.parametrize("sizes", SIZES)
@pytest.mark.parametrize("nproj", [5, 16, 20])
@pytest.mark.parametrize("disjoint", [True, False])
def test_nonlocal_matches_dense(sizes, nproj, disjoint):
    from lynx_amd import _lib as L, core
    s = System(N, np.array([6.0, 5.8, 5.5]), np.array([[0.3, 0.4, 0.5]]), with_nonlocal=False)
    lens = np.sqrt((s.latvec ** 2).sum(axis=1))
    raw, images, displ, gamma = raw_projectors(nproj, sizes, disjoint, 7, lens)
    dv = abs(np.linalg.det(s.latvec)) / s.nd
    op = s.oracle_op()
    H0 = s.hamiltonian()                       # builds s.core
    lat, grid, st, dom, halo = s.core
    H = core.Hamiltonian(0).setup(st, dom, grid, halo, core.NonlocalProjector().setup_raw(**raw))
    kpt = tuple(2 * np.pi * np.array([0.2, -0.3, 0.15]) / lens)
    lib = L.lib()
    lo, hi = s.veff.min() - 2.0, 60.0
    lc = lo + 0.3 * (hi - lo)

    def ref_apply(x, k, c):
        op.set_kpoint(k)
        y = op.apply(x, s.veff, c=c)
        alpha = np.zeros((displ[-1], x.shape[1]), x.dtype)
        ph = [np.exp(-1j * np.dot(k, R)) if np.iscomplexobj(x) else 1.0 for _, _, _, R in images]
        for (a, g, ch, _), p in zip(images, ph):
            alpha[displ[a]:displ[a + 1]] += p * (ch.T @ x[g])
        alpha *= dv * gamma[:, None]
        for (a, g, ch, _), p in zip(images, ph):
            y[g] += np.conj(p) * (ch @ alpha[displ[a]:displ[a + 1]])
        return y

    def ref_filter(x, k):
        e, c = (hi - lc) / 2, (hi + lc) / 2
        s1 = sg = e / (lo - c)
        old, y = x, ref_apply(x, k, -c) * (sg / e)
        for _ in range(DEG - 1):
            t = 1 / (2 / s1 - sg)
            old, y = y, ref_apply(y, k, -c) * (2 * t / e) - sg * t * old
            sg = t
        return y

    H.set_veff(s.veff)
    for dt, ncols in ((np.float64, (1, 15, 17)), (np.complex128, (1, 8, 9)), (np.float32, (16,)),
                      (np.complex64, (7,))):
        cplx = np.dtype(dt).kind == "c"
        single = np.dtype(dt).itemsize == (8 if cplx else 4)
        wide = complex if cplx else float
        k = kpt if cplx else (0.0, 0.0, 0.0)
        H.set_kpoint(k)
        blocks = [s.random_block(n, 20 + n, cplx).astype(dt) for n in ncols]
        refs = [ref_filter(x.astype(wide), k) for x in blocks]
        for x, rf in zip(blocks, refs):
            ref = ref_apply(x.astype(wide), k, -0.3)
            got = H._apply(x.T.copy(), s.veff, -0.3, dt).reshape(x.shape[1], -1).T
            assert rel(got, ref) < (5e-6 if single else 1e-12), (dt, x.shape)
            y, xf = np.zeros_like(x, order="F"), np.asfortranarray(x)
            for _ in range(3):                 # direct, captured and replayed
                y[:] = 0
                L.check(lib.lynx_cheb_filter(H.ctx, L.dtype_code(dt), L.vptr(xf), s.nd, L.vptr(y), s.nd, x.shape[1],
                                             DEG, lc, lo, hi, L.MEM_HOST), H.ctx)
                assert rel(y, rf) < (5e-5 if single else 1e-11), (dt, x.shape)
        bf = core.BatchFilter([(H, k)] * len(blocks))
        for _ in range(2):
            for got, rf in zip(bf.filter(blocks, DEG, lc, lo, hi, dtype=dt), refs):
                assert rel(got, rf) < (5e-5 if single else 1e-11), dt
        bf.close()

    # bfloat16 storage
    H.set_kpoint((0.0, 0.0, 0.0))
    xb = np.asfortranarray(bf16_round(s.random_block(18, 3)))
    x = (xb.astype(np.uint32) << 16).view(np.float32).astype(float)
    yb = np.zeros_like(xb, order="F")
    L.check(lib.lynx_cheb_filter(H.ctx, L.BF16, L.vptr(xb), s.nd, L.vptr(yb), s.nd, 18, DEG, lc, lo, hi, L.MEM_HOST),
            H.ctx)
    y = (yb.astype(np.uint32) << 16).view(np.float32)
    assert rel(y, ref_filter(x, (0.0, 0.0, 0.0))) < 2e-2
    del H0
