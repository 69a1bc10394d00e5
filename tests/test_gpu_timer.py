"""The kernel event timer (mlg_timer_read) on the transform launches: one
record per launch, with the launch's own bytes as work, whichever kernel a
length takes."""
import numpy as np
import pytest

from mlegs_amd import hip as H
from mlegs_amd.configs import CFG1

pytestmark = pytest.mark.gpu


def grid(**k):
    return H.Grid(dict(CFG1, **dict(dict(nr=24, nth=4, nx=4, nrchop=12, ntchop=2, nxchop=2), **k)))


# the four-step kernels, the theta lines, the short, mixed-radix and direct lengths
@pytest.mark.parametrize("n", [8, 64, 512, 12, 24, 46, 1024])
def test_one_record_per_transform(n):
    g = grid(nth=n)
    f = g.scalar(H.PPP, np.ones(g.shape(H.PPP), dtype=complex))
    g.timer(True)
    H.horfft(f, -1)
    H.horfft(f, 1)
    g.timer(False)
    for k in ("horfft_fwd", "horfft_bwd"):
        assert g.timer_read(k)[1:] == (1, 16.0 * 24 * 4 * (n + 2), "byte")
    g.close()
    g = grid(nx=n)
    f = g.scalar(H.FFF, np.zeros(g.shape(H.FFF), dtype=complex))
    H.rtran(f, 1)
    g.timer(True)
    H.verfft(f, 1)
    H.verfft(f, -1)
    g.timer(False)
    for k in ("verfft_fwd", "verfft_bwd"):
        assert g.timer_read(k)[1:] == (1, 16.0 * 24 * 2 * (n + 3), "byte")
    g.close()
