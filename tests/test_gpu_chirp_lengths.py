"""Chirp-z windows in the whole-signal kernel over the transform lengths that its cost
rule picks: lengths a few points from each other that take other plans, the ends of
the workgroup shapes, lengths that leave a CU one workgroup or two. Against the
oracle's long-double DFT, with the tolerance of the transforms of any length."""
import numpy as np
import pytest

import oracle as O
from henon_map_cpp_amd import _capi as C
from test_gpu_fft_any import quasi_periodic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [53, 107, 113, 281, 302, 317, 499, 509, 607, 639, 853, 1021, 1277, 1283, 1538, 1571, 1685,
                               1733, 1779, 1852, 1996, 2081, 2497, 2507, 2521, 2543, 2557, 2707, 3279, 4999, 5113])
def test_chirp_lengths_match_oracle_dft(N):
    n = 1 if N > 1000 else 3
    h = quasi_periodic(N, n, seed=N + 5)
    rows = np.ascontiguousarray(h.transpose(2, 1, 0))
    got = C.history_tunes(C.DeviceBuffer.from_array(rows), n, N, [(0, N - 1)], "fft", row_len=N)
    for i in range(n):
        want = [O.fft_tune(h[:, 0, i], h[:, 1, i]), O.fft_tune(h[:, 2, i], h[:, 3, i])]
        np.testing.assert_allclose(got[0, :, i], want, rtol=0, atol=1e-12, err_msg=f"N={N} particle {i}")
