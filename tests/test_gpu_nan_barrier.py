"""No point is inside a NaN barrier: every particle is lost in the turn it starts
with, as the oracle has it, whatever the number of turns and whichever kernel runs
them (tracking forward and inverse, batched jobs, the adjoint's forward sweep)."""
import numpy as np
import pytest
import torch

import oracle as O
from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import adjoint as A
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu
TURNS = [1, 7, 8, 9, 100, 1000]
NAN = float("nan")


def lattice(T):
    wx, wy = C.sps_modulation(0.168, 16.0, 0, T), C.sps_modulation(0.201, 16.0, 0, T)
    return O.Tables(wx, wy), C.DeviceBuffer.from_array(C.build_table(wx, wy))


def oracle_track(x0, tables, T, inverse):
    p = O.Particles(*x0)
    p.steps[:] = T if inverse else 0
    O.lib().or_track(*p.state(), p.n, *tables.ptrs(), T, 0.5, NAN, np.nan, int(inverse), 1)
    return p.x, p.px, p.y, p.py, p.steps


@pytest.mark.parametrize("T", TURNS)
def test_every_particle_is_lost_at_once(T):
    x0 = W.ball(200, 0.2, seed=3)
    tables, tab = lattice(T)
    for mode in (C.MODE_EXACT, C.MODE_FAST):
        for inverse in (False, True):
            want = oracle_track(x0, tables, T, inverse)
            assert np.isnan(want[0]).all() and np.all(want[4] == (T if inverse else 0))
            dev = C.DeviceParticles(*x0, steps=np.full(200, T if inverse else 0, dtype=np.uint32))
            C.track(dev, tab, T, T, 0.5, NAN, inverse, mode)
            for u, v in zip(want, dev.get()):
                assert np.array_equal(u, v, equal_nan=True)
        dev = C.DeviceParticles(*x0)
        C.track_batch([(dev, tab, T, T, 0.5, NAN)], mode)
        for u, v in zip(oracle_track(x0, tables, T, False), dev.get()):
            assert np.array_equal(u, v, equal_nan=True)


@pytest.mark.parametrize("T", TURNS)
def test_adjoint_forward_parks_every_particle_at_once(T):
    x0 = torch.from_numpy(np.stack(W.ball(200, 0.2, seed=3))).cuda()
    for mode in ("exact", "fast"):
        st, birk, alive, ck = A.OrbitAdjoint(T, 0.168, 0.201, 16.0, 0.5, NAN, every=8, mode=mode).forward(x0)
        assert not bool(alive.any()) and bool(torch.isnan(st).all()) and bool(torch.isnan(birk).all())
        # the checkpoints after the first hold the parked points
        assert torch.equal(ck[0], x0) and bool((ck[1:] == 0).all())
