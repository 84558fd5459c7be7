"""The Lanczos bounds do not depend on what their scratch vectors held before:
a run on a potential of NaN leaves NaN in them, and the next run on the same
context gives the bounds of a fresh context, bit for bit."""
import numpy as np
import pytest

from systems import A_SI, DIAMOND, System

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
def test_lanczos_ignores_old_scratch(cplx):
    import ctypes

    from lynx_amd import _lib as L
    s = System((12, 12, 12), A_SI, DIAMOND)
    H = s.hamiltonian()

    def bounds(veff):
        H.set_veff(veff)
        lo, hi, it = ctypes.c_double(), ctypes.c_double(), ctypes.c_int()
        L.check(L.lib().lynx_lanczos_bounds(H.ctx, L.C128 if cplx else L.F64, ctypes.byref(lo), ctypes.byref(hi), 1e-2,
                                            1000, 1, ctypes.byref(it)), H.ctx)
        return lo.value, hi.value, it.value

    want = bounds(s.veff)
    assert np.isfinite(want).all()
    bounds(np.full_like(s.veff, np.nan))
    assert bounds(s.veff) == want
