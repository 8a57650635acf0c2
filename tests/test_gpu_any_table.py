"""Tables whose records are not rotations: losses are found on the turn they happen,
as the oracle has them, and points that such a table brings down to where products
leave the normal range keep the reference's roundings. A gain on one record, on all
from some turn on, or on all, at turn counts and places around the windows of 64
records; tracking both ways and both modes, batched jobs, the adjoint's forward
sweep."""
import numpy as np
import pytest
import torch

import oracle as O
from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import adjoint as A
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu
MU, BARRIER = 0.5, 3.0


def lattice(T, gains):
    """gains: [(first, last, plane, factor)] on the sines and cosines."""
    t = O.Tables(C.sps_modulation(0.168, 16.0, 0, T), C.sps_modulation(0.201, 16.0, 0, T))
    pairs = ((t.sx, t.cx), (t.sy, t.cy))
    for first, last, plane, factor in gains:
        for a in pairs[plane]:
            a[first:last] *= factor
    return t, np.ascontiguousarray(np.stack([t.sx, t.cx, t.sy, t.cy], axis=1))


def oracle_track(x0, tables, T, inverse=False):
    p = O.Particles(*x0)
    p.steps[:] = T if inverse else 0
    O.lib().or_track(*p.state(), p.n, *tables.ptrs(), T, MU, BARRIER, np.nan, int(inverse), 1)
    return p.x, p.px, p.y, p.py, p.steps


def same(a, b):
    for u, v, name in zip(a, b, ["x", "px", "y", "py", "steps"]):
        assert np.array_equal(u, v, equal_nan=True), name


CASES = [(T, [(k, k + 1, plane, f)])
         for T, k in [(40, 1), (40, 6), (40, 39), (200, 63), (200, 64), (200, 65), (200, 131), (130, 129)]
         for plane, f in [(0, 40.0), (1, 9.0)]]
CASES += [(200, [(0, 200, 0, 1.01)]), (200, [(90, 200, 1, 1.02), (0, 90, 1, 0.99)]), (300, [(65, 300, 0, 1e3)]),
          (900, [(0, 900, 0, 0.4), (0, 900, 1, 0.5)]), (900, [(70, 900, 0, 0.3), (70, 900, 1, 0.4)])]


@pytest.mark.parametrize("T,gains", CASES)
def test_losses_and_roundings_with_any_table(T, gains):
    x0 = np.stack(W.ball(200, 0.3, seed=17))
    tables, tab = lattice(T, gains)
    tdev = C.DeviceBuffer.from_array(tab)
    for inverse in (False, True):
        want = oracle_track(x0, tables, T, inverse)
        for mode in (C.MODE_EXACT, C.MODE_FAST):
            steps = np.full(200, T if inverse else 0, dtype=np.uint32)
            dev = C.DeviceParticles(*x0, steps=steps)
            C.track(dev, tdev, T, T, MU, BARRIER, inverse, mode)
            got = dev.get()
            if mode == C.MODE_EXACT:
                same(want, got)
            one = C.DeviceParticles(*x0, steps=steps)  # every turn of one-turn calls is tested
            for _ in range(T):
                C.track(one, tdev, T, 1, MU, BARRIER, inverse, mode)
            same(one.get(), got)
    dev = C.DeviceParticles(*x0)
    C.track_batch([(dev, tdev, T, T, MU, BARRIER)], C.MODE_EXACT)
    same(oracle_track(x0, tables, T), dev.get())
    adj = A.OrbitAdjoint(T, 0.168, 0.201, 16.0, MU, BARRIER, every=8)
    adj.table = torch.from_numpy(tab).cuda()
    st, birk, alive, ck = adj.forward(torch.from_numpy(x0).cuda())
    want = oracle_track(x0, tables, T)
    same(want[:4], st.cpu().numpy())
    assert np.array_equal(alive.cpu().numpy() == 1, want[4] == T)
    # checkpoints: the state at each interval's start, the origin once lost
    for q in range(ck.shape[0]):
        at = oracle_track(x0, tables, 8 * q) if q else [*x0]
        assert np.array_equal(ck[q].cpu().numpy(), np.nan_to_num(np.stack(at[:4]), nan=0.0))
