"""The MEGNO takes ratios of norms only: a start matrix times a power of two, which
leaves every mantissa in place, gives the same MEGNO bit for bit, at any scale, with
and without renormalisation and construct windows, in one launch and across
segments; a scale that is no power of two moves it by roundings alone."""
import numpy as np
import pytest

from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu


def megno(n, T, scale, renorm, mode=C.MODE_EXACT, **kw):
    wx, wy = (C.sps_modulation(q, 16.0, 0, T) for q in (0.168, 0.201))
    tab = C.DeviceBuffer.from_array(C.build_table(wx, wy))
    return C.track_indicators(C.DeviceParticles(*W.ball(n, 0.2, seed=7)), tab, T, T, 0.5, 10.0, mode, renorm,
                              [1, T // 3, T - 1, T], matrix=np.tile(np.eye(4) * scale, (n, 1, 1)), **kw)["megno"]


@pytest.mark.parametrize("n,T", [(193, 300), (52_003, 1300)])
@pytest.mark.parametrize("renorm", [0, 37])
def test_powers_of_two_change_nothing(n, T, renorm):
    base = megno(n, T, 1.0, renorm)
    assert np.isfinite(base).all()
    for e in (-300, -41, 40, 400):
        assert np.array_equal(megno(n, T, 2.0 ** e, renorm), base)
    assert np.array_equal(megno(n, T, 2.0 ** 40, renorm, megno_birkhoff=[T // 2]),
                          megno(n, T, 1.0, renorm, megno_birkhoff=[T // 2]))


def test_other_scales_move_roundings_alone():
    """The matrix products round at 2^-53 of their size, which a change of mantissa
    redraws at every turn: by turn k the norm's logarithm has moved by about sqrt(k)
    of them, MEGNO(300) by a few 1e-15 times that; held to 1e-13."""
    base = megno(193, 300, 1.0, 0)
    for scale in (1e120, 1e-120, 3.0):
        np.testing.assert_allclose(megno(193, 300, scale, 0), base, rtol=0, atol=1e-13)
