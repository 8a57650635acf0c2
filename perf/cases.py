"""Performance cases: the work a user of the tracker has it do, through the package's entry points.

    listed()            the cases with a name
    draw(rng)           one more case of the same ranges, without a name
    prepare(case, seed) what a program holds before the call: initial conditions, tracker or device table
    run(state)          one pass; returns every output of the call
    work(case)          bytes and FP64 operations that one pass cannot do without (`live`: share of the particle-turns
                        before losses, measured for the listed cases)
    exact(case, seed)   the same outputs from plain numpy / torch in float64, or None where that takes too long

Kinds of case (`kind`):
    track         tracking with loss; `host` true: the drop-in call on numpy arrays (upload, track, read back),
                  false: particles and table resident on the GPU, the C entry point on the caller's stream
    reversibility forward and back again, error at two turn counts (the inverse map)
    indicators    tangent map + MEGNO + FLI (+ Birkhoff windows) in one call
    tunes         tune_all: trajectory, Birkhoff and FFT tunes of four windows
    adjoint       whole-orbit gradients: forward sweep with checkpoints and backward sweep
    batch         many uneven jobs in one call, 30 % of them with the MEGNO
    constructs    the per-turn construct classes driven from Python, as the reference's notebooks do
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import henon_map_cpp_amd as hm
from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import adjoint as A

QX, QY = 0.168, 0.201           # tunes of the dynamic-aperture scans
BARRIER = math.sqrt(10.0)       # loss at r^2 >= 10
LINES = (1, 2, 3, 6, 7, 10, 12)  # multiples of 1 / 868.12 turns in the modulation spectrum


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: a few orbits looked at interactively
        dict(name="track_64_orbits", kind="track", n=64, turns=100, grid=False, radius=0.3, mu=0.2, eps=16.0,
             mode="exact", host=True, live=1.0),
        # the reference's dynamic-aperture scan of one parameter set: 100 x 100 grid, no modulation, no octupole
        dict(name="da_scan_100", kind="track", n=10_000, turns=10_000, grid=True, radius=0.6, mu=0.0, eps=0.0,
             mode="exact", host=True, live=0.64),
        # the large modulated scan: 1000 x 1000 grid, 1e5 turns, resident particles
        dict(name="da_scan_1000", kind="track", n=1_000_000, turns=100_000, grid=True, radius=0.6, mu=0.5, eps=32.0,
             mode="exact", host=False, live=0.56),
        # statistics over a random ensemble in the fast arithmetic, any particle count
        dict(name="ensemble_fast", kind="track", n=300_007, turns=20_000, grid=False, radius=0.5, mu=-0.37, eps=8.0,
             mode="fast", host=False, live=0.97),
        # reversibility error of a middle-sized set (inverse map)
        dict(name="reversibility", kind="reversibility", n=20_000, turns=2_000, radius=0.4, mu=0.5, eps=32.0,
             mode="exact"),
        # the chaos-indicator workload: 131072 particles x 1e5 turns
        dict(name="indicators_131072", kind="indicators", n=131_072, turns=100_000, radius=0.5, mu=0.5, eps=32.0,
             renorm=100, windows=0, mode="exact"),
        # a small set with tune diffusion from two Birkhoff windows, exact orbit
        dict(name="indicators_windows", kind="indicators", n=4_099, turns=3_000, radius=0.35, mu=0.3, eps=8.0,
             renorm=100, windows=2, mode="exact_orbit"),
        # the reference's tune notebook: 90000 particles, 1e4 turns, windows [0, 500], [500, 1000]
        dict(name="tunes_notebook", kind="tunes", n=90_000, turns=10_000, window=500, radius=0.2, mu=0.0, eps=0.0),
        # tunes of a smaller modulated set over windows of a length that is not round
        dict(name="tunes_odd", kind="tunes", n=3_001, turns=2_090, window=811, radius=0.4, mu=0.25, eps=16.0),
        # gradients of an orbit loss, 65536 particles x 1e4 turns, default checkpoint interval
        dict(name="adjoint_65536", kind="adjoint", n=65_536, turns=10_000, every=0, radius=0.4, mu=0.5, eps=16.0,
             mode="exact"),
        # uneven independent jobs in one call
        dict(name="batch_192", kind="batch", jobs=192, n_max=16_384, t_max=50_000),
        # constructs driven turn by turn: many small calls
        dict(name="constructs_1000", kind="constructs", n=1_000, turns=40, radius=0.3, mu=0.5, eps=16.0),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi], odd ones among them."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["track", "track", "track", "reversibility", "indicators", "indicators", "tunes", "tunes",
                       "adjoint", "batch", "constructs"])
    eps = rng.choice([0.0, round(rng.uniform(1.0, 64.0), 3)])
    mu = rng.choice([0.0, 0.25, 0.5, 0.75, 1.0, round(rng.uniform(-1.0, 1.0), 4)])
    if kind == "track":
        host = rng.random() < 0.5
        n = _log(rng, 64, 100_000 if host else 1_000_000)
        grid = rng.random() < 0.5
        if grid:
            n = max(8, math.isqrt(n)) ** 2
        turns = _log(rng, 100, min(100_000, 20_000_000_000 // n))
        return dict(kind=kind, n=n, turns=turns, grid=grid, radius=0.6 if grid else round(rng.uniform(0.2, 0.6), 3),
                    mu=mu, eps=eps, mode=rng.choice(["exact", "exact", "fast"]), host=host, live=0.7)
    if kind == "reversibility":
        return dict(kind=kind, n=_log(rng, 100, 100_000), turns=_log(rng, 200, 10_000),
                    radius=round(rng.uniform(0.2, 0.5), 3), mu=mu, eps=eps, mode=rng.choice(["exact", "fast"]))
    if kind == "indicators":
        n = _log(rng, 500, 131_072)
        return dict(kind=kind, n=n, turns=_log(rng, 300, min(50_000, 1_500_000_000 // n)),
                    radius=round(rng.uniform(0.2, 0.45), 3), mu=mu, eps=eps, renorm=rng.choice([0, 10, 100, 100, 250]),
                    windows=rng.choice([0, 0, 1, 2]), mode=rng.choice(["exact", "exact", "exact_orbit"]))
    if kind == "tunes":
        n = _log(rng, 200, 60_000)
        turns = _log(rng, 256, min(10_000, 400_000_000 // n))
        return dict(kind=kind, n=n, turns=turns, window=_log(rng, 50, turns // 2),
                    radius=round(rng.uniform(0.1, 0.4), 3), mu=mu, eps=eps)
    if kind == "adjoint":
        n = _log(rng, 200, 65_536)
        return dict(kind=kind, n=n, turns=_log(rng, 100, 10_000), every=rng.choice([0, 0, 8, 64, 256]),
                    radius=round(rng.uniform(0.2, 0.4), 3), mu=mu, eps=eps, mode="exact")
    if kind == "batch":
        return dict(kind=kind, jobs=_log(rng, 8, 256), n_max=_log(rng, 1_000, 16_384), t_max=_log(rng, 2_000, 50_000))
    return dict(kind=kind, n=_log(rng, 64, 20_000), turns=rng.randint(10, 40), radius=round(rng.uniform(0.2, 0.4), 3),
                mu=mu, eps=eps)


# ------------------------------------------------------------------ inputs
def _ball(n, radius, rng):
    """n points of the 4D ball, uniform in its volume."""
    d = rng.normal(size=(n, 4))
    d *= (radius * rng.uniform(size=n) ** 0.25 / np.linalg.norm(d, axis=1))[:, None]
    return [np.ascontiguousarray(d[:, k]) for k in range(4)]


def _points(case, seed):
    rng = np.random.default_rng([seed, 1])
    if case.get("grid"):
        side = math.isqrt(case["n"])
        v = np.linspace(0.0, case["radius"] * rng.uniform(0.95, 1.05), side + 1)[1:]
        xx, yy = np.meshgrid(v, v)
        return [xx.ravel().copy(), np.zeros(case["n"]), yy.ravel().copy(), np.zeros(case["n"])]
    return _ball(case["n"], case["radius"], rng)


def _spectrum(seed):
    """Line coefficients (sum 1e-4, as the SPS lines' scale) and angular frequencies."""
    a = np.random.default_rng([seed, 2]).uniform(0.1, 1.0, len(LINES))
    return a / a.sum() * 1e-4, np.array([m * (2 * math.pi / 868.12) for m in LINES])


def _tracker(case, seed, turns):
    coef, freq = _spectrum(seed)
    return hm.henon_tracker(turns, QX, QY, "custom", epsilon=case["eps"], coefficients=coef, frequencies=freq)


def _batch_jobs(case, seed):
    """(n, turns, tune x, tune y, eps, mu, MEGNO) of every job: sizes by the case, lattices by the seed."""
    rng = np.random.default_rng([case["jobs"], case["n_max"], case["t_max"]])
    lattice = np.random.default_rng([seed, 3])
    out = []
    for k in range(case["jobs"]):
        n = int(round(math.exp(rng.uniform(math.log(64), math.log(case["n_max"])))))
        t = int(round(math.exp(rng.uniform(math.log(1_000), math.log(case["t_max"])))))
        if k == 0:
            n, t = case["n_max"] // 2, case["t_max"]  # the longest job is always there
        out.append((n, t, *lattice.uniform(0.15, 0.32, 2), lattice.uniform(0.0, 64.0), lattice.uniform(-1.0, 1.0),
                    k % 10 < 3))
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "batch":
        coef, freq = _spectrum(seed)
        jobs = _batch_jobs(case, seed)
        total = sum(j[0] for j in jobs)
        s["x0"] = torch.from_numpy(np.stack(_ball(total, 0.6, np.random.default_rng([seed, 1])))).cuda()
        s["tables"] = [torch.from_numpy(C.build_table(C.lines_modulation(qx, eps, coef, freq, 0, t),
                                                      C.lines_modulation(qy, eps, coef, freq, 0, t))).cuda()
                       for n, t, qx, qy, eps, mu, megno in jobs]
        s["jobs"] = jobs
        return s
    x0 = _points(case, seed)
    if kind == "track" and not case["host"]:
        coef, freq = _spectrum(seed)
        T = case["turns"]
        s["x0"] = torch.from_numpy(np.stack(x0)).cuda()
        s["table"] = torch.from_numpy(C.build_table(C.lines_modulation(QX, case["eps"], coef, freq, 0, T),
                                                    C.lines_modulation(QY, case["eps"], coef, freq, 0, T))).cuda()
        return s
    if kind == "adjoint":
        coef, freq = _spectrum(seed)
        s["x0"] = torch.from_numpy(np.stack(x0)).cuda()
        s["adjoint"] = A.OrbitAdjoint(case["turns"], QX, QY, case["eps"], case["mu"], BARRIER, coef=coef, freq=freq,
                                      every=case["every"] or None, mode=case["mode"])
        return s
    s["x0"] = x0
    s["tracker"] = _tracker(case, seed, case["turns"] + 1)
    if kind == "indicators":
        s["samples"], s["windows"] = _samples(case), _windows(case)
    return s


def _samples(case):
    """Turn counts at which MEGNO and FLI are recorded: a tenth, all."""
    return [max(1, case["turns"] // 10), case["turns"]]


def _windows(case):
    """Birkhoff windows over the first and the second half."""
    h = case["turns"] // 2
    return [(0, h), (h, case["turns"])][:case["windows"]]


# ------------------------------------------------------------------ one pass
def _state(p):
    return [np.asarray(p.get_x()), p.get_px(), p.get_y(), p.get_py(), p.get_steps()]


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def run(state):
    case = state["case"]
    return _RUN[case["kind"]](state, case)


def _run_track(s, case):
    if case["host"]:
        p = hm.particles(*s["x0"])
        s["tracker"].track(p, case["turns"], case["mu"], BARRIER, mode=case["mode"])
        return _state(p)
    x = s["x0"].clone()
    steps = torch.zeros(x.shape[1], dtype=torch.int32, device="cuda")
    C.check(C.lib().hm_track(*(x[k].data_ptr() for k in range(4)), steps.data_ptr(), x.shape[1],
                             s["table"].data_ptr(), s["table"].shape[0], case["turns"], case["mu"], BARRIER,
                             float("nan"), 0, C.MODE_FAST if case["mode"] == "fast" else C.MODE_EXACT, None,
                             _stream()))
    return [x, steps]


def _run_reversibility(s, case):
    p = hm.particles(*s["x0"])
    err = s["tracker"].reversibility_error(p, [case["turns"] // 10, case["turns"]], case["mu"], BARRIER,
                                           mode=case["mode"])
    return [err, *_state(p)]


def _run_indicators(s, case):
    p = hm.particles(*s["x0"])
    d = s["tracker"].tangent_indicators(p, case["turns"], case["mu"], BARRIER, renorm_every=case["renorm"],
                                        samples=s["samples"], birkhoff=s["windows"], mode=case["mode"])
    kinds = ("megno", "fli", "matrix", "log_scale") + (("birkhoff",) if s["windows"] else ())
    return {**{k: d[k] for k in kinds}, "steps": p.get_steps()}


def _run_tunes(s, case):
    # the tracker's own call, whose arrays tune_all puts into a DataFrame: all four windows
    w = case["window"]
    p = hm.particles(*s["x0"])
    birkhoff, fft = s["tracker"].tracker.all_tunes(p.particles, case["turns"], case["mu"], BARRIER, float("nan"),
                                                   False, [0, w], [w, 2 * w])
    return [birkhoff, fft]


def _run_adjoint(s, case):
    adj = s["adjoint"]
    st, birk, alive, ck = adj.forward(s["x0"])
    # loss: mean final r^2 plus mean Birkhoff average of x^2 over the survivors
    ok = alive.bool()
    m = ok.sum().clamp(min=1).to(torch.float64)
    seed_state = torch.where(ok[None, :], 2.0 * st / m, torch.zeros_like(st))
    seed_birk = torch.where(ok, 1.0 / m, torch.zeros_like(birk))
    gx, gp = adj.backward(ck, alive, seed_state, seed_birk)
    return [st, birk, alive, gx, gp]


def _run_batch(s, case):
    x = s["x0"].clone()
    steps = torch.zeros(x.shape[1], dtype=torch.int32, device="cuda")
    megno = torch.zeros(x.shape[1], dtype=torch.float64, device="cuda")
    arr = (C.Job * len(s["jobs"]))()
    at = 0
    for k, ((n, t, qx, qy, eps, mu, meg), tab) in enumerate(zip(s["jobs"], s["tables"])):
        arr[k] = C.Job(*(x[c, at:].data_ptr() for c in range(4)), steps[at:].data_ptr(), n, tab.data_ptr(), t, t, 100,
                       mu, BARRIER, float("nan"), megno[at:].data_ptr() if meg else None)
        at += n
    C.check(C.lib().hm_track_batch(arr, len(s["jobs"]), C.MODE_EXACT, None, _stream()))
    return [x, steps, megno]


def _run_constructs(s, case):
    n, T, mu, t = case["n"], case["turns"], case["mu"], s["tracker"]
    p = hm.particles(*s["x0"])
    a, b = hm.matrix_4d_vector(n), hm.matrix_4d_vector(n)
    v = hm.vector_4d(np.tile([1.0, 0.0, 0.0, 0.0], (n, 1)))
    megno, lyap = hm.megno_construct(n), hm.lyapunov_birkhoff_construct(n, T)
    tune = hm.tune_birkhoff_construct(n, [T // 2])
    tune.first_add(p)
    one = hm.matrix_4d_vector(n)
    for _ in range(T):
        b.explicit_copy(a)
        one.set_with_tracker(t, p, mu)
        a.structured_multiply(t, p, mu)
        v.multiply(one)
        lyap.add(v)
        v.normalize()
        megno.add(a, b)
        t.track(p, 1, mu, BARRIER)
        tune.add(p)
    return [megno.get_values(), lyap.get_values_b(), np.asarray(tune.get_tune1_x()), np.asarray(tune.get_tune2_y()),
            a.get_matrix(), v.get_vectors(), *_state(p)]


_RUN = dict(track=_run_track, reversibility=_run_reversibility, indicators=_run_indicators, tunes=_run_tunes,
            adjoint=_run_adjoint, batch=_run_batch, constructs=_run_constructs)


# ------------------------------------------------------------------ work
def _map_flops(mu):
    """One turn of one particle; an FMA counts 2."""
    return 40.0 if mu else 26.0


def work(case):
    kind = case["kind"]
    if kind == "batch":
        jobs = _batch_jobs(case, 0)
        return {"bytes": sum(72.0 * j[0] + 32.0 * j[1] for j in jobs),
                "flops": sum(0.8 * j[0] * j[1] * (40.0 + (138.0 if j[6] else 0.0)) for j in jobs)}
    n, T = case["n"], case["turns"]
    m = _map_flops(case["mu"])
    if kind == "track":
        return {"bytes": 68.0 * n + 32.0 * T, "flops": case["live"] * n * T * m}
    if kind == "reversibility":
        return {"bytes": 48.0 * n + 32.0 * T, "flops": n * (T + T + T // 10) * m}
    if kind == "indicators":
        return {"bytes": n * (32.0 + 136.0 + 32.0 + 16.0 * case["windows"]) + 40.0 * T,
                "flops": n * T * (m + 138.0)}
    if kind == "tunes":
        # each window's signal once per plane: an FFT, and 8 operations and an angle per sample
        lens = [case["window"] + 1, case["window"] + 1, T + 1, T]
        fft = sum(5.0 * v * math.log2(v) for v in lens)
        return {"bytes": n * (32.0 + 2 * 8.0 * 8) + 32.0 * T, "flops": n * (T * m + 2 * fft + 2 * 8.0 * sum(lens[:3]))}
    if kind == "adjoint":
        return {"bytes": n * (32.0 + 32.0 + 8.0 + 1.0 + 32.0 + 8.0 + 64.0) + 72.0 * T, "flops": n * T * (m + 109.0)}
    return {"bytes": n * (32.0 + 36.0 + 128.0 + 64.0) + 32.0 * T, "flops": n * T * (m + 250.0)}


# ------------------------------------------------------------------ in 64 bits, without the package
def _omegas(tune, eps, seed, turns):
    coef, freq = _spectrum(seed)
    w = []
    for i in range(turns):
        total = 0.0
        for c, f in zip(coef, freq):
            total += float(c) * math.cos(float(f) * i)
        w.append(2 * math.pi * tune * (1 + eps * total))
    return w


def _records(case, seed, turns):
    wx, wy = _omegas(QX, case["eps"], seed, turns), _omegas(QY, case["eps"], seed, turns)
    return [(math.sin(a), math.cos(a), math.sin(b), math.cos(b)) for a, b in zip(wx, wy)]


def _kick(x, y, mu):
    kx, ky = (x * x) - (y * y), (-2.0 * x) * y
    ox = mu * (((x * x) * x) - (((3.0 * y) * y) * x))
    oy = mu * (((y * y) * y) - (((3.0 * x) * x) * y))
    return kx, ky, ox, oy


def _forward(z, mu, rec):
    x, px, y, py = z
    sx, cx, sy, cy = rec
    kx, ky, ox, oy = _kick(x, y, mu)
    px, py = px + kx, py + ky
    if mu != 0.0:
        px, py = px + ox, py + oy
    return [(x * cx) + (px * sx), ((-x) * sx) + (px * cx), (y * cy) + (py * sy), ((-y) * sy) + (py * cy)]


def _backward(z, mu, rec):
    x, px, y, py = z
    sx, cx, sy, cy = rec
    x, px, y, py = (x * cx) - (px * sx), (x * sx) + (px * cx), (y * cy) - (py * sy), (y * sy) + (py * cy)
    kx, ky, ox, oy = _kick(x, y, mu)
    if mu != 0.0:
        px, py = px - ox, py - oy
    return [x, px - kx, y, py - ky]


def _lose(z, steps, up):
    """Loss at the barrier: every coordinate NaN, the turn not counted."""
    r2 = ((z[0] * z[0]) + (z[1] * z[1])) + ((z[2] * z[2]) + (z[3] * z[3]))
    ok = r2 < BARRIER * BARRIER
    steps += up * ok
    if not ok.all():
        for c in z:
            c[~ok] = np.nan
    return z


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch" or case.get("mode") == "fast" and kind != "adjoint":
        return None  # too long; and of a chaotic orbit in another rounding only the first turns
    n, T = case["n"], case["turns"]
    per_turn = dict(track=40, reversibility=90, indicators=250, tunes=120, adjoint=0, constructs=400)[kind]
    if per_turn * T * (1.5e-6 + 1.2e-9 * n) > 10.0 or kind == "adjoint" and (n * T > 400_000 or T > 1_500):
        return None
    with np.errstate(all="ignore"):
        return _EXACT[kind](case, seed)


def _exact_track(case, seed):
    z, steps = _points(case, seed), np.zeros(case["n"], dtype=np.int64)
    for rec in _records(case, seed, case["turns"]):
        z = _lose(_forward(z, case["mu"], rec), steps, 1)
    if case["host"]:
        return [*z, steps]
    return [np.stack(z), steps.astype(np.int32)]


def _exact_reversibility(case, seed):
    T, mu = case["turns"], case["mu"]
    z0 = _points(case, seed)
    recs = _records(case, seed, T)
    z, steps, out = [c.copy() for c in z0], np.zeros(case["n"], dtype=np.int64), []
    for k in range(T):
        z = _lose(_forward(z, mu, recs[k]), steps, 1)
        if k + 1 in (T // 10, T):
            b = [c.copy() for c in z]
            for j in range(k, -1, -1):
                b = _lose(_backward(b, mu, recs[j]), steps.copy(), -1)
            out.append(np.sqrt(sum((u - v) * (u - v) for u, v in zip(b, z0))))
    return [np.stack(out), *z, steps]


def _jacobian(x, y, mu, rec):
    sx, cx, sy, cy = rec
    mu3, mu6 = mu * 3, mu * 6
    a = ((2.0 * x) + ((mu3 * x) * x)) - ((mu3 * y) * y)
    b = (-2.0 * y) - ((mu6 * x) * y)
    o = np.zeros_like(x)
    f = np.full_like
    return [[cx + sx * a, f(x, sx), sx * b, o], [-sx + cx * a, f(x, cx), cx * b, o],
            [sy * b, o, cy - sy * a, f(x, sy)], [cy * b, o, -sy - cy * a, f(x, cy)]]


def _product(j, m):
    """Structured J M, M as [4][4][n]."""
    r = np.empty_like(m)
    r[0] = ((j[0][0] * m[0]) + (j[0][1] * m[1])) + (j[0][2] * m[2])
    r[1] = ((j[1][0] * m[0]) + (j[1][1] * m[1])) + (j[1][2] * m[2])
    r[2] = ((j[2][0] * m[0]) + (j[2][2] * m[2])) + (j[2][3] * m[3])
    r[3] = ((j[3][0] * m[0]) + (j[3][2] * m[2])) + (j[3][3] * m[3])
    return r


def _weights(n):
    t = np.arange(n) / n
    with np.errstate(all="ignore"):
        w = np.exp(-1 / (t * (1.0 - t)))
    return w / w.sum()


def _exact_indicators(case, seed):
    n, T, mu = case["n"], case["turns"], case["mu"]
    z, steps = _points(case, seed), np.zeros(n, dtype=np.int64)
    m = np.tile(np.eye(4)[:, :, None], (1, 1, n))
    scale = np.zeros(n)  # log10 of the scale taken out of m
    norm = np.log10((m * m).sum(axis=(0, 1))) * 0.5
    l1, l2 = np.zeros(n), np.zeros(n)
    megno, fli = [], []
    wins = [(a, b, _weights(b - a), np.zeros((2, n))) for a, b in _windows(case)]
    angle = (np.arctan2(z[1], z[0]), np.arctan2(z[3], z[2])) if wins else None
    for k, rec in enumerate(_records(case, seed, T)):
        m = _product(_jacobian(z[0], z[2], mu, rec), m)
        z = _lose(_forward(z, mu, rec), steps, 1)
        m[:, :, np.isnan(z[0])] = np.nan
        # MEGNO by the constructs' recursion, on the logarithm of the norm
        now = np.log10((m * m).sum(axis=(0, 1))) * 0.5
        l1 = l1 + (now - norm) * (k + 1)
        l2 = l2 + l1 / (k + 1)
        norm = now
        if k + 1 in _samples(case):
            megno.append(l2 / (k + 1))
            fli.append((scale + np.log10(np.sqrt((m[:, 0] * m[:, 0]).sum(axis=0)))) / (k + 1))
        if case["renorm"] and (k + 1) % case["renorm"] == 0:
            f = np.sqrt((m * m).sum(axis=(0, 1)))
            ok = ~np.isnan(f)
            m[:, :, ok] = m[:, :, ok] * (1.0 / f[ok])
            scale[ok] = scale[ok] + np.log10(f[ok])
            norm = np.log10((m * m).sum(axis=(0, 1))) * 0.5
        if wins:
            new = (np.arctan2(z[1], z[0]), np.arctan2(z[3], z[2]))
            for p in range(2):
                d = new[p] - angle[p]
                d = np.where(d < 0.0, d + 2 * math.pi, d)
                for a, b, w, acc in wins:
                    if a < k + 1 <= b:
                        acc[p] += w[k - a] * d
            angle = new
    out = {"megno": np.stack(megno), "fli": np.stack(fli), "matrix": np.ascontiguousarray(m.transpose(2, 0, 1)),
           "log_scale": scale, "steps": steps}
    if wins:
        out["birkhoff"] = np.stack([1.0 - w[3] / (2 * math.pi) for w in wins])
    return out


def _fft_tune(c):
    """Interpolated position of the spectrum's first maximum, c as [signals][N] complex."""
    N = c.shape[1]
    s = np.abs(np.fft.fft(c * (2 * np.sin(math.pi * np.arange(N) / N) ** 2), axis=1))
    k = s.argmax(axis=1)
    i = np.arange(len(k))
    down = s[i, k - 1] > s[i, (k + 1) % N]
    lo = np.where(down, k - 1, k)
    a, b, q = s[i, lo], s[i, (lo + 1) % N], math.cos(2 * math.pi / N)
    root = np.sqrt(q * q * ((a + b) * (a + b)) - 2 * a * b * (2 * (q * q) - q - 1))
    amp = (-(a + b * q) * (a - b) + b * root) / ((a * a) + (b * b) + 2 * a * b * q)
    tune = np.abs(1.0 - (lo / N + np.arcsin(amp * math.sin(2 * math.pi / N)) / (2 * math.pi)))
    return np.where(k == 0, 1.0, np.where(k == N - 1, 0.0, tune))


def _exact_tunes(case, seed):
    n, T, w = case["n"], case["turns"], case["window"]
    z, steps = _points(case, seed), np.zeros(n, dtype=np.int64)
    h = np.empty((4, T + 1, n))
    h[:, 0] = z
    for k, rec in enumerate(_records(case, seed, T)):
        z = _lose(_forward(z, case["mu"], rec), steps, 1)
        h[:, k + 1] = z
    h = h - h.mean(axis=1, keepdims=True)
    lost = np.isnan(h).any(axis=(0, 1))
    h = np.ascontiguousarray(np.where(lost, 0.0, h).transpose(0, 2, 1))
    birk, fft = [], []
    for a, b, first in ((0, w, 0), (w, 2 * w, w), (0, T, 0), (0, T, 1)):  # the last FFT takes samples 1..T
        wt = _weights(b - a)
        for p in range(2):
            th = np.arctan2(h[2 * p + 1, :, a:b + 1], h[2 * p, :, a:b + 1])
            d = np.diff(th, axis=1)
            d = np.where(d < 0.0, d + 2 * math.pi, d)
            birk.append(np.where(lost, np.nan, 1.0 - (d * wt).sum(axis=1) / (2 * math.pi)))
            fft.append(np.where(lost, np.nan, _fft_tune(h[2 * p, :, first:b + 1] + 1j * h[2 * p + 1, :, first:b + 1])))
    return [np.stack(birk, axis=1), np.stack(fft, axis=1)]


def _exact_adjoint(case, seed):
    """Reverse mode by torch on the CPU, the lattice parameters as one value per particle."""
    n, T = case["n"], case["turns"]
    coef, freq = _spectrum(seed)
    x0 = torch.from_numpy(np.stack(_points(case, seed))).requires_grad_()
    one = torch.ones(n, dtype=torch.float64)
    eps, mu = (one * case["eps"]).requires_grad_(), (one * case["mu"]).requires_grad_()
    wx, wy = (one * (2 * math.pi * QX)).requires_grad_(), (one * (2 * math.pi * QY)).requires_grad_()
    weights = _weights(T)
    x, px, y, py = x0
    birk = torch.zeros(n, dtype=torch.float64)
    alive = torch.ones(n, dtype=torch.bool)
    for k in range(T):
        line = sum(float(c) * math.cos(float(f) * k) for c, f in zip(coef, freq))
        a, b = wx * (1 + eps * line), wy * (1 + eps * line)
        px = px + (x * x - y * y) + mu * (x * x * x - 3.0 * y * y * x)
        py = py - 2.0 * x * y + mu * (y * y * y - 3.0 * x * x * y)
        x, px = x * a.cos() + px * a.sin(), px * a.cos() - x * a.sin()
        y, py = y * b.cos() + py * b.sin(), py * b.cos() - y * b.sin()
        ok = alive & ((x * x + px * px + y * y + py * py).detach() < BARRIER * BARRIER)
        if not bool(ok.all()):
            x, px, y, py = (torch.where(ok, v, torch.zeros_like(v)) for v in (x, px, y, py))
        alive = ok
        birk = birk + float(weights[k]) * x * x
    st = torch.stack([x, px, y, py])
    if case["mu"] == 0.0 or not bool(alive.all()):
        return None  # lost points have their own conventions
    loss = (st * st).sum() / n + birk.sum() / n
    gx, ge, gm, ga, gb = torch.autograd.grad(loss, [x0, eps, mu, wx, wy])
    return [st.detach(), birk.detach(), alive.to(torch.uint8), gx, torch.stack([ge, gm, ga, gb])]


def _exact_constructs(case, seed):
    n, T, mu = case["n"], case["turns"], case["mu"]
    z, steps = _points(case, seed), np.zeros(n, dtype=np.int64)
    m = np.tile(np.eye(4)[:, :, None], (1, 1, n))
    v = np.zeros((4, n))
    v[0] = 1.0
    l1, l2, l3, lyap, t1, t2 = (np.zeros(n) for _ in range(6))
    w, half = _weights(T), _weights(T // 2)
    norm = 0.5 * np.log10((m * m).sum(axis=(0, 1)))
    angle = np.arctan2(z[1], z[0]), np.arctan2(z[3], z[2])
    for k, rec in enumerate(_records(case, seed, T)):
        j = _jacobian(z[0], z[2], mu, rec)
        m = _product(j, m)
        v = np.stack([sum(j[r][c] * v[c] for c in range(4)) for r in range(4)])
        f = np.sqrt((v * v).sum(axis=0))
        lyap = lyap + np.log(f) * w[k]
        v = v / f
        now = 0.5 * np.log10((m * m).sum(axis=(0, 1)))
        l1 = l1 + (now - norm) * (k + 1)
        l2 = l2 + l1 / (k + 1)
        l3 = l2 / (k + 1)
        norm = now
        z = _lose(_forward(z, mu, rec), steps, 1)
        new = np.arctan2(z[1], z[0]), np.arctan2(z[3], z[2])
        d = [np.where(b - a > 0, b - a, b - a + 2 * math.pi) for a, b in zip(angle, new)]
        angle = new
        if k + 1 < T // 2:
            t1 = t1 + d[0] * half[k + 1]
        elif k + 1 < 2 * (T // 2):
            t2 = t2 + d[1] * half[k + 1 - T // 2]
    return [l3, lyap, t1[None], t2[None], np.ascontiguousarray(m.transpose(2, 0, 1)), np.ascontiguousarray(v.T), *z, steps]


_EXACT = dict(track=_exact_track, reversibility=_exact_reversibility, indicators=_exact_indicators,
              tunes=_exact_tunes, adjoint=_exact_adjoint, constructs=_exact_constructs)
