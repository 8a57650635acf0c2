"""Barriers and octupole strengths so large that a turn's reach overflows: the loss is
found in the turn where the oracle finds it, also when that turn is a call's last
(no radius is safe for a turn that goes untested then, or a small one is)."""
import numpy as np
import pytest

import oracle as O
from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("barrier", [1e95, 1e120, np.inf])
@pytest.mark.parametrize("mu", [1e9, -1e20, 1e60])
def test_losses_fall_in_the_oracle_turn(mu, barrier):
    scale = np.abs(mu) ** -0.5
    x0 = [v * scale * np.geomspace(0.1, 10.0, 256) for v in W.ball(256, 1.0, seed=8)]
    for T in (8, 9, 16, 24, 64):
        wx, wy = C.sps_modulation(0.168, 16.0, 0, T), C.sps_modulation(0.201, 16.0, 0, T)
        tables, tab = O.Tables(wx, wy), C.DeviceBuffer.from_array(C.build_table(wx, wy))
        p = O.Particles(*x0)
        O.lib().or_track(*p.state(), p.n, *tables.ptrs(), T, mu, barrier, np.nan, 0, 1)
        for every in (0, 8):
            dev = C.DeviceParticles(*x0)
            C.track(dev, tab, T, T, mu, barrier, cfg=C.LaunchCfg(0, every, 0, 0))
            for u, v in zip((p.x, p.px, p.y, p.py, p.steps), dev.get()):
                assert np.array_equal(u, v, equal_nan=True)
    assert len(np.unique(p.steps)) > 5
