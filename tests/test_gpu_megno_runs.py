"""The MEGNO sums over straight runs of plain turns taken two at a time: run
lengths of both parities (renormalisation intervals, neighbouring samples, turn
counts around the first segment), every mode, single calls and batched jobs, and
tangent matrices that start at zero or far from 1."""
import os

import numpy as np
import pytest

import oracle as O
from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu
NT = min(os.cpu_count() or 1, 16)


def setup(T, n=193, r=0.35, seed=31):
    coef, freq = W.seeded_line_coefficients(), W.line_frequencies()
    wx, wy = (C.lines_modulation(q, 16.0, coef, freq, 0, T) for q in (0.168, 0.201))
    return O.Tables(wx, wy), C.DeviceBuffer.from_array(C.build_table(wx, wy)), W.ball(n, r, seed=seed)


@pytest.mark.parametrize("mode", [C.MODE_EXACT, C.MODE_EXACT_ORBIT, C.MODE_FAST])
@pytest.mark.parametrize("T,renorm", [(1, 0), (2, 1), (3, 2), (124, 0), (125, 3), (126, 7), (127, 100), (377, 10),
                                      (1003, 101)])
def test_megno_runs_of_both_parities(T, renorm, mode):
    ot, tdev, x0 = setup(T)
    samples = sorted({1, 2, max(1, T // 2), max(1, T // 2 + 1), max(1, T - 1), T} & set(range(1, T + 1)))
    got = C.track_indicators(C.DeviceParticles(*x0), tdev, T, T, 0.5, 10.0, mode, renorm, samples, matrix=True)
    want = O.indicators(O.Particles(*x0), ot, T, 0.5, 10.0, renorm, samples, n_threads=NT)
    # fused products and maps agree with the unfused ones on regular orbits only
    tol = dict(rtol=1e-12, atol=1e-13) if mode == C.MODE_EXACT else dict(rtol=1e-9, atol=1e-10)
    ok = slice(None) if mode == C.MODE_EXACT else np.all(np.abs(want["megno"]) < 2.5, axis=0)
    for key in ("megno", "fli"):
        np.testing.assert_allclose(got[key][:, ok], want[key][:, ok], equal_nan=True, **tol)
    if mode == C.MODE_EXACT:
        assert np.array_equal(got["matrix"], want["matrix"], equal_nan=True)
    if mode != C.MODE_EXACT_ORBIT and T > 1:
        megno = C.DeviceBuffer(8 * len(x0[0]))
        C.track_batch([(C.DeviceParticles(*x0), tdev, T, T, 0.5, 10.0, megno, renorm)], mode)
        assert np.array_equal(megno.download(np.float64, len(x0[0])), got["megno"][-1], equal_nan=True)


def test_megno_of_scaled_and_zero_start_matrices():
    T, samples = 200, [1, 60, 199, 200]
    ot, tdev, x0 = setup(T, r=0.2)
    n = len(x0[0])
    eye = np.tile(np.eye(4), (n, 1, 1))

    def megno(matrix, **kw):
        return C.track_indicators(C.DeviceParticles(*x0), tdev, T, T, 0.5, 10.0, C.MODE_EXACT, 0, samples,
                                  matrix=matrix, **kw)["megno"]

    base = megno(eye)
    assert np.isfinite(base).all()
    # only ratios of norms enter: powers of two leave every rounding but the
    # logarithm's in place (|log10| up to 150, so 150 2^-53 times a few)
    for e in (-500, -40, 40, 500):
        np.testing.assert_allclose(megno(eye * 2.0 ** e), base, rtol=0, atol=1e-12)
    # the logarithm of a zero norm: no MEGNO, with and without construct windows
    assert np.isnan(megno(eye * 0.0)).all()
    assert np.isnan(megno(eye * 0.0, megno_birkhoff=[50])).all()
