"""The passes of the whole-signal transforms against the oracle's long-double DFT:
every register radix (2 to 13 and 16), prime passes on the matrix cores with full
and ragged tiles (19 x 23, 53 x 61, 19 x 151, 73 x 137 points) and on the vector
units (17^3, a 37 near the most points of its shape), the most points of each
workgroup shape and the next length, chirp-z lengths; and a spectrum that is zero
everywhere, whose first maximum is entry 0. The tolerance is that of the transforms
of any length: both round a tune of a quasi-periodic signal at 1e-13 or so."""
import numpy as np
import pytest

import oracle as O
from henon_map_cpp_amd import _capi as C
from test_gpu_fft_any import quasi_periodic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [9, 11, 13, 18, 77, 96, 143, 432, 437, 640, 641, 720, 1029, 1280, 1281, 1716, 2187, 2560,
                               2574, 2869, 3233, 4608, 4913, 5120, 5148, 8192, 9360, 9361, 9990, 10001, 10140])
def test_passes_match_oracle_dft(N):
    n = 1 if N > 1000 else 4
    h = quasi_periodic(N, n, seed=N + 21)
    rows = np.ascontiguousarray(h.transpose(2, 1, 0))
    major = C.history_tunes(C.DeviceBuffer.from_array(np.ascontiguousarray(h)), n, N, [(0, N - 1)], "fft")
    got = C.history_tunes(C.DeviceBuffer.from_array(rows), n, N, [(0, N - 1)], "fft", row_len=N)
    assert np.array_equal(major, got)
    for i in range(n):
        want = [O.fft_tune(h[:, 0, i], h[:, 1, i]), O.fft_tune(h[:, 2, i], h[:, 3, i])]
        np.testing.assert_allclose(got[0, :, i], want, rtol=0, atol=1e-12, err_msg=f"N={N} particle {i}")


@pytest.mark.parametrize("N", [10, 437, 501, 10000])
def test_zero_spectrum_takes_entry_zero(N):
    d = C.DeviceBuffer.from_array(np.zeros((N, 4, 2)))
    assert np.all(C.history_tunes(d, 2, N, [(0, N - 1)], "fft") == 1.0)
