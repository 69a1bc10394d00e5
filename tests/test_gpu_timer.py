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
@pytest.mark.parametrize("n", [8, 64, 512, 12, 30, 46, 1024])
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


def rows(cfg, nrchop):
    return sum(max(0, min(nrchop, nrchop - m)) for m in range(cfg["ntchop"]))


def force_flop(cfg):
    """RTRAN backward of the right-hand side: nine fields, W's at NRCHOP and the others at NRCHOP + 3."""
    return 2.0 * cfg["nr"] * (2 * cfg["nxchop"] - 1) * (8 * rows(cfg, cfg["nrchop"] + 3) + rows(cfg, cfg["nrchop"]))


@pytest.mark.parametrize("split", [0, 1])
def test_work_of_the_right_hand_side(split):
    cfg = dict(CFG1, nr=32, nth=16, nx=16, nrchop=22, ntchop=6, nxchop=5, split=split)
    g = H.Grid(cfg)
    f = [g.scalar(H.FFF, np.zeros(g.shape(H.FFF), dtype=complex)) for _ in range(6)]
    g.timer(True)
    H.calc_boussi_force(*f)
    g.timer(False)
    assert g.timer_read("rtran_bwd")[2] == force_flop(cfg)
    p = [g.scalar(H.PPP, np.ones(g.shape(H.PPP), dtype=complex)) for _ in range(7)]
    g.timer(True)
    H.vdotpsub(*p)
    g.timer(False)
    assert g.timer_read("products")[1:] == (1, 16.0 * 32 * 16 * 16 * 7, "byte")
    g.close()


def test_work_of_a_sweep():
    cfgs = [dict(CFG1, nr=32, nth=16, nx=16, nrchop=22, ntchop=6, nxchop=5),
            dict(CFG1, nr=48, nth=32, nx=16, nrchop=32, ntchop=11, nxchop=5)]
    runs = []
    for c in cfgs:
        g = H.Grid(c)
        s, f = H.Solver(g), [g.scalar(H.FFF, np.zeros(g.shape(H.FFF), dtype=complex)) for _ in range(3)]
        s.initialize(*f)
        runs.append((s, *f))
    sw = H.Sweep(runs, grouped=True, tune=False)
    sw.steps(2)
    assert sw.info()["grouped_gflop_per_step"] == pytest.approx(1e-9 * sum(map(force_flop, cfgs)), rel=1e-12)
    sw.close()
