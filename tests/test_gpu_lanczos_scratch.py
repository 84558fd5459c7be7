"""The Lanczos bounds do not depend on what the memory of their scratch vectors
held before: device memory of their size is filled with NaN and freed just
before a context takes its own.  Bar against a context without that: the tuner
may pick another launch shape, which changes the rounding only (1e-9)."""
import ctypes

import numpy as np
import pytest

from systems import A_SI, DIAMOND, System

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
def test_lanczos_ignores_old_memory(cplx):
    from lynx_amd import _lib as L
    from lynx_amd.hipmem import DeviceArray
    s = System((12, 12, 12), A_SI, DIAMOND)
    size = s.nd * (16 if cplx else 8)

    def bounds(poison):
        H = s.hamiltonian()
        H.set_veff(s.veff)
        old = [DeviceArray(size) for _ in range(poison)]
        for d in old:
            d.fill_bytes(0xff)
        for d in old:
            d.free()
        lo, hi, it = ctypes.c_double(), ctypes.c_double(), ctypes.c_int()
        L.check(L.lib().lynx_lanczos_bounds(H.ctx, L.C128 if cplx else L.F64, ctypes.byref(lo), ctypes.byref(hi), 1e-2,
                                            1000, 1, ctypes.byref(it)), H.ctx)
        return np.array([lo.value, hi.value])

    want, got = bounds(0), bounds(64)
    assert np.isfinite(want).all() and want[0] < want[1]
    assert np.abs(got - want).max() < 1e-9 * np.abs(want).max()


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_bounds_of_an_operator_that_is_not_finite(cplx, bad):
    # a projector whose energy is no number: no bounds, where a NaN used to
    # end the iteration as converged
    from lynx_amd import _lib as L, core
    s = System((12, 12, 12), A_SI, DIAMOND, with_nonlocal=False)
    s.hamiltonian()
    lat, grid, st, dom, halo = s.core
    raw = dict(img_atom=[0], img_ndc=[5], img_nproj=[1], gpos=np.arange(5), chi=np.ones(5),
               img_shift=np.zeros(3), n_atom=1, ip_displ=[0, 1])
    for gamma in (bad, 0.5):
        H = core.Hamiltonian(0).setup(st, dom, grid, halo,
                                      core.NonlocalProjector().setup_raw(**raw, gamma=np.array([gamma])))
        H.set_veff(s.veff)
        lo, hi = ctypes.c_double(7.0), ctypes.c_double(7.0)
        got = L.lib().lynx_lanczos_bounds(H.ctx, L.C128 if cplx else L.F64, ctypes.byref(lo), ctypes.byref(hi), 1e-2,
                                          1000, 1, None)
        if gamma == 0.5:
            assert got == L.OK and lo.value < hi.value
        else:
            assert got == L.E_NONFINITE and lo.value == hi.value == 7.0
