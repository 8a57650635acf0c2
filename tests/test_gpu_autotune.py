"""hm_track without a configuration runs the one that hm_autotune_track remembered:
as many launches as its segments, for a set small enough to go in one launch by
default; and one again once it is forgotten."""
import numpy as np
import pytest

from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu
T = 3000


def segments(every):
    done, length, count = 0, min(125, every), 0
    while done < T:
        done, length, count = done + length, min(2 * length, every), count + 1
    return count


def launches(x0, tab):
    p = C.DeviceParticles(*x0)
    C.profile_reset()
    C.profile_enable(True)
    try:
        C.track(p, tab, T, T, 0.5, 3.0, False, C.MODE_EXACT)
        return C.profile_read("k_track")[1], p.get()
    finally:
        C.profile_enable(False)
        C.profile_reset()


@pytest.mark.parametrize("n", [500, 14_400])
def test_remembered_segments_are_used(n):
    wx, wy = (C.sps_modulation(q, 16.0, 0, T) for q in (0.168, 0.201))
    tab = C.DeviceBuffer.from_array(C.build_table(wx, wy))
    x0 = W.ball(n, 0.3, seed=4)
    try:
        C.check(C.lib().hm_autotune_clear())
        before, want = launches(x0, tab)
        best, _ = C.autotune_track(C.DeviceParticles(*x0), tab, T, 0.5, 3.0, warm_turns=200, trial_turns=800)
        tuned, got = launches(x0, tab)
    finally:
        C.check(C.lib().hm_autotune_clear())
    after, _ = launches(x0, tab)
    assert before == after == 1
    assert tuned == segments(best.compact_every) > 1
    assert all(np.array_equal(a, b, equal_nan=True) for a, b in zip(want, got))
