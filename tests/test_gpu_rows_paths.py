"""Trajectory rows by the wave-uniform path and the per-lane path against the
sample-major history, bit for bit: turn counts around the groups of 16 samples and
the pairs of records, losses at every turn, particles NaN from the start, wavefronts
with a particle that holds one NaN coordinate or another turn index (per-lane path),
a turn index that leaves the table, inverse tracking, records that are not finite."""
import numpy as np
import pytest

from henon_map_cpp_amd import _capi as C
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("turns", [0, 1, 14, 15, 16, 17, 31, 32, 47, 64, 129])
@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("mu", [0.0, 0.37])
def test_rows_equal_history(turns, inverse, mu):
    n, slots = 64 * 5 + 9, turns + 40
    coef, freq = W.seeded_line_coefficients(), W.line_frequencies()
    tab = C.build_table(C.lines_modulation(0.168, 32.0, coef, freq, 0, slots),
                        C.lines_modulation(0.201, 32.0, coef, freq, 0, slots))
    tab[20 if inverse else turns + 5, 1] = np.nan  # reached by some wavefronts only
    dev = C.DeviceBuffer.from_array(tab)
    x0 = np.stack(W.ball(n, 0.9, seed=turns + 1))
    x0[:, 3::50] = np.nan
    x0[2, 64 + 7] = np.nan                      # second wavefront: held coordinates
    steps = np.full(n, turns + 30 if inverse else 0)
    steps[128:192] += 7                         # third: another index, all the same
    steps[192 + 5] += 1                         # fourth: one particle apart
    if inverse:
        steps[256:320] = 3                      # fifth: leaves the table
    else:
        steps[256:320] = slots - 3
    a, b = C.DeviceParticles(*x0, steps=steps), C.DeviceParticles(*x0, steps=steps)
    rows, means = C.track_rows(a, dev, slots, turns, mu, 1.6, inverse, means=True)
    fa = C.take_status()
    hist = C.track_history(b, dev, slots, turns, mu, 1.6, inverse)
    assert fa == C.take_status()
    L = C.row_length(turns)
    got = rows.download(np.float64, n * 4 * L).reshape(n, 4, L)
    want = hist.download(np.float64, (turns + 1) * 4 * n).reshape(turns + 1, 4, n)
    assert np.array_equal(got[:, :, :turns + 1], want.transpose(2, 1, 0), equal_nan=True)
    assert np.array_equal(got[:, :, turns + 1:], np.repeat(got[:, :, turns:turns + 1], L - turns - 1, axis=2),
                          equal_nan=True)
    s = np.zeros((4, n))
    for m in range(turns + 1):
        s = s + want[m]
    assert np.array_equal(means.download(np.float64, 4 * n).reshape(4, n), s / (turns + 1), equal_nan=True)
    for u, v in zip(a.get(), b.get()):
        assert np.array_equal(u, v, equal_nan=True)
