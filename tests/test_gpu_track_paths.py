"""Ways that hm_track still has of running the same turns, against each other bit for
bit in both modes and directions: workgroups of 64, 192 and 256 threads; one launch
against segments; wavefronts whose particles share a turn index (records by scalar
loads, turns in pairs) against those whose particles do not (a record per lane)."""
import numpy as np
import pytest

from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu
T, LEN = 611, 640


def table():
    coef, freq = W.seeded_line_coefficients(), W.line_frequencies()
    return C.DeviceBuffer.from_array(C.build_table(*(C.lines_modulation(q, 32.0, coef, freq, 0, LEN)
                                                     for q in (0.168, 0.201))))


def run(tab, x0, steps, mode, inverse, cfg=None):
    p = C.DeviceParticles(*x0, steps=steps)
    C.track(p, tab, LEN, T, 0.4, 3.0, inverse, mode, cfg)
    assert C.take_status() == 0
    return p.get()


@pytest.mark.parametrize("mode", [C.MODE_EXACT, C.MODE_FAST])
@pytest.mark.parametrize("inverse", [False, True])
def test_blocks_segments_and_lanes_agree(mode, inverse):
    tab, n = table(), 5003
    x0 = np.stack(W.ball(n, 0.7, seed=6))
    x0[:, ::211] = np.nan
    first = T + 5 if inverse else 3
    steps = np.full(n, first, dtype=np.uint32)
    want = run(tab, x0, steps, mode, inverse)
    lost = np.isnan(want[0]).mean()
    assert 0.1 < lost < 0.9
    for cfg in (C.LaunchCfg(64, -1, 0, 0), C.LaunchCfg(256, -1, 0, 0), C.LaunchCfg(192, 100, 0, 0),
                C.LaunchCfg(64, 7, 0, 0), C.LaunchCfg(256, 1000, 0, 0)):
        for a, b in zip(run(tab, x0, steps, mode, inverse, cfg), want):
            assert np.array_equal(a, b, equal_nan=True)
    # every other particle a turn later: no wavefront shares its turn index
    mixed = steps + (np.arange(n) % 2).astype(np.uint32)
    later = run(tab, x0, steps + np.uint32(1), mode, inverse)
    for got, a, b in zip(run(tab, x0, mixed, mode, inverse), want, later):
        assert np.array_equal(got[::2], a[::2], equal_nan=True)
        assert np.array_equal(got[1::2], b[1::2], equal_nan=True)
