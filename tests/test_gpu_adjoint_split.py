"""The backward sweep of few particles runs its two chains in two wavefronts, that of
more in one. A particle's gradients do not depend on which: a set large enough for
one must equal its halves, each small enough for two, bit for bit, over turn counts
with a short last chunk or a single one, checkpoint intervals from one chunk on,
windows of segments, lost particles and particles NaN from the start."""
import numpy as np
import pytest
import torch

from henon_map_cpp_amd import adjoint as A
from henon_map_cpp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("turns,every,scratch", [(300, 64, None), (301, 64, None), (307, 8, None), (300, 16, "one"),
                                                 (5, 8, None), (16, 16, None), (264, 88, None)])
@pytest.mark.parametrize("mode,mu", [("exact", 0.5), ("exact", 0.0), ("fast", 0.37)])
def test_halves_equal_the_whole(turns, every, scratch, mode, mu, monkeypatch):
    n, half = 36_003, 18_100
    x0 = np.stack(W.ball(n, 0.8, seed=5))
    x0[:, ::501] = np.nan
    x0 = torch.from_numpy(x0).cuda()
    if scratch:
        monkeypatch.setenv("HM_ADJOINT_SCRATCH_BYTES", "1")  # one segment a window
    adj = A.OrbitAdjoint(turns, 0.168, 0.201, 16.0, mu, 2.0, every=every, mode=mode)
    g = torch.Generator().manual_seed(9)
    seed_s = torch.randn((4, n), generator=g, dtype=torch.float64).cuda()
    seed_b = torch.randn((n,), generator=g, dtype=torch.float64).cuda()

    def run(sl):
        st, birk, alive, ck = adj.forward(x0[:, sl].contiguous())
        gx, gp = adj.backward(ck, alive, seed_s[:, sl].contiguous(), seed_b[sl].contiguous())
        return [v.cpu().numpy() for v in (st, birk[None], alive[None], gx, gp)]

    whole = run(slice(0, n))
    parts = [run(slice(k, min(k + half, n))) for k in range(0, n, half)]
    for k, v in enumerate(whole):
        assert np.array_equal(v, np.concatenate([p[k] for p in parts], axis=1), equal_nan=True), k
    assert 0.0 < whole[2].mean() < 1.0
