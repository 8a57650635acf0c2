"""The gradients follow one order of operations: each turn of the adjoint as written
out below (every fused multiply-add in its place, the kick's partial derivatives one
by one) gives the device's gradients bit for bit, whichever kernel sweeps."""
import ctypes
import ctypes.util

import numpy as np
import pytest
import torch

import oracle as O
from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import adjoint as A
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu

_libm = ctypes.CDLL(ctypes.util.find_library("m"))
_libm.fma.restype = ctypes.c_double
_libm.fma.argtypes = [ctypes.c_double] * 3
fma = np.vectorize(_libm.fma, otypes=[np.float64])


def host_gradients(states, table, dtable, weights, mu, seed_s, seed_b):
    """states: [T + 1][4][n]; returns grad_x0, grad_params, both [4][n]."""
    lx, lpx, ly, lpy = (v.copy() for v in seed_s)
    n = lx.size
    g_eps, g_mu, g_wx, g_wy = (np.zeros(n) for _ in range(4))
    bseed, mu3, mu6 = 2.0 * seed_b, 3.0 * mu, 6.0 * mu
    for k in range(len(states) - 2, -1, -1):
        pre, post = states[k], states[k + 1]
        sx, cx, sy, cy = table[k]
        dt = dtable[k]
        lx = fma(bseed * weights[k], post[0], lx)
        dwx = fma(lx, post[1], -lpx * post[0])
        dwy = fma(ly, post[3], -lpy * post[2])
        g_wx = fma(dwx, dt[0], g_wx)
        g_wy = fma(dwy, dt[2], g_wy)
        g_eps = fma(dwx, dt[1], fma(dwy, dt[3], g_eps))
        lxt, lpt = fma(cx, lx, -sx * lpx), fma(sx, lx, cx * lpx)
        lyt, lqt = fma(cy, ly, -sy * lpy), fma(sy, ly, cy * lpy)
        x, y = pre[0], pre[2]
        xx, yy = x * x, y * y
        if mu != 0.0:
            g_mu = fma(lpt, x * fma(-3.0, yy, xx), fma(lqt, y * fma(-3.0, xx, yy), g_mu))
        ja = fma(mu3, xx - yy, 2.0 * x)
        jb = fma(-mu6 * x, y, -2.0 * y)
        lx, ly = fma(ja, lpt, fma(jb, lqt, lxt)), fma(jb, lpt, fma(-ja, lqt, lyt))
        lpx, lpy = lpt, lqt
    return np.stack([lx, lpx, ly, lpy]), np.stack([g_eps, g_mu, g_wx, g_wy])


# 7: k_adjoint_sweep; 8 and 32: two wavefronts for few particles, one for many
@pytest.mark.parametrize("every,copies", [(7, 1), (8, 1), (32, 1), (32, 1700)])
@pytest.mark.parametrize("mu", [0.5, 0.37, 0.0])
def test_gradients_equal_the_turns_written_out(every, copies, mu):
    turns, n = 61, 24
    coef, freq = C.sps_lines()
    adj = A.OrbitAdjoint(turns, 0.168, 0.201, 16.0, mu, 10.0, every=every)
    wx = C.lines_modulation(0.168, 16.0, coef, freq, 0, turns)
    wy = C.lines_modulation(0.201, 16.0, coef, freq, 0, turns)
    x0 = np.stack(W.ball(n, 0.3, seed=3))
    rng = np.random.default_rng(8)
    seed_s, seed_b = rng.normal(size=(4, n)), rng.normal(size=n)
    tracker, p = O.Tracker.from_tables(O.Tables(wx, wy)), O.Particles(*x0)
    states = [np.stack([p.x, p.px, p.y, p.py])]
    for _ in range(turns):
        tracker.track(p, 1, mu, barrier=10.0, n_threads=1)
        states.append(np.stack([p.x, p.px, p.y, p.py]))
    want = host_gradients(states, C.build_table(wx, wy), adj.dtable.cpu().numpy(), adj.weights.cpu().numpy(), mu,
                          seed_s, seed_b)

    def many(v):
        return torch.as_tensor(np.tile(v, copies)).cuda()

    st, _, alive, ck = adj.forward(many(x0))
    got = adj.backward(ck, alive, many(seed_s), many(seed_b))
    assert bool(alive.all()) and torch.equal(st, many(states[-1]))
    for a, b in zip(got, want):
        assert np.array_equal(a.cpu().numpy(), np.tile(b, copies))
