"""Calls of few wavefronts run all turns in one launch, larger ones in segments with
loss compaction between them. A particle's results do not depend on which: a set
large enough for segments must equal its parts, each small enough for one launch,
bit for bit, over losses in every segment, particles NaN from the start and particles
with one NaN coordinate."""
import numpy as np
import pytest

from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu

T = 1700


def table():
    coef, freq = W.seeded_line_coefficients(), W.line_frequencies()
    return C.DeviceBuffer.from_array(C.build_table(C.lines_modulation(0.168, 32.0, coef, freq, 0, T),
                                                   C.lines_modulation(0.201, 32.0, coef, freq, 0, T)))


def points(n):
    x0 = np.stack(W.ball(n, 0.75, seed=3))
    x0[:, ::997] = np.nan
    x0[1, 5::1009] = np.nan
    return x0


@pytest.mark.parametrize("mode", [C.MODE_EXACT, C.MODE_FAST])
@pytest.mark.parametrize("inverse", [False, True])
def test_track_segments_equal_one_launch(mode, inverse):
    tab, n, part = table(), 70_001, 33_000

    def run(x0):
        p = C.DeviceParticles(*x0, steps=np.full(x0.shape[1], T if inverse else 0))
        C.track(p, tab, T, T, 0.4, 3.0, inverse, mode)
        return np.stack([np.asarray(v, dtype=np.float64) for v in p.get()])

    x0 = points(n)
    whole = run(x0)
    parts = np.concatenate([run(x0[:, k:k + part]) for k in range(0, n, part)], axis=1)
    assert np.array_equal(whole, parts, equal_nan=True)
    assert C.take_status() == 0


@pytest.mark.parametrize("extra", [{}, {"birkhoff": [(0, 900), (800, T)]},
                                   {"birkhoff": [(3, T)], "megno_birkhoff": [400, 1600], "tune_birkhoff": [700]}])
def test_indicator_segments_equal_one_launch(extra):
    tab, n, part = table(), 52_003, 26_010

    def run(x0):
        p = C.DeviceParticles(*x0)
        r = C.track_indicators(p, tab, T, T, 0.4, 3.0, mode=C.MODE_EXACT, renorm_every=100, samples=[200, T],
                               matrix=True, **extra)
        out = {k: np.asarray(v) for k, v in r.items() if v is not None and np.asarray(v).size}
        return out, [np.asarray(v) for v in p.get()]

    x0 = points(n)
    whole, state = run(x0)
    runs = [run(x0[:, k:k + part]) for k in range(0, n, part)]
    for c, v in enumerate(state):
        assert np.array_equal(v, np.concatenate([s[c] for _, s in runs]), equal_nan=True)
    for name, v in whole.items():
        axis = 0 if name in ("matrix", "log_scale") else v.ndim - 1
        assert np.array_equal(v, np.concatenate([o[name] for o, _ in runs], axis=axis), equal_nan=True), name
    assert C.take_status() == 0
