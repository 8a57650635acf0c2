"""FFT tunes of signals with infinite samples (infinite, so not cut out as lost ones
are): the spectrum's first entry is NaN then, a scan for the first maximum from there
on never leaves it, and entry 0 gives the tune 1. Lengths of every kind of plan:
radices in registers, prime passes on the matrix cores and on the vector units, powers
of two, chirp-z, the transforms through memory."""
import numpy as np
import pytest

from henon_map_cpp_amd import _capi as C

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [15, 17, 19, 38, 53, 96, 100, 107, 500, 501, 1000, 2048, 2187, 4096, 5000, 8192, 10000, 10001,
                               12000])
def test_an_infinite_sample_gives_entry_zero(N):
    L = C.row_length(N - 1)
    rows = np.random.default_rng(N).normal(size=(3, 4, L)) * 0.1
    rows[0, 1, 1] = np.inf           # px: infinite in the imaginary part of the signal
    rows[1, 2, 1] = -np.inf          # y: in the real part
    rows[2, 0, N // 2] = np.inf      # x: X_0 = inf - inf
    rows[2, 0, N // 3] = -np.inf
    got = C.history_tunes(C.DeviceBuffer.from_array(rows), 3, N, [(0, N - 1)], "fft", row_len=L,
                          means=C.DeviceBuffer.from_array(np.zeros((4, 3))))[0]
    assert got[0, 0] == got[1, 1] == got[0, 2] == 1.0
    for plane, particle in ((1, 0), (0, 1), (1, 2)):
        assert 0.0 <= got[plane, particle] <= 1.0
