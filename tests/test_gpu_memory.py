"""Device memory that a call leaves with the context's pool, in fields (arrays
of the largest space), and the diagnostics against the oracle where their
fields are taken to PFF a group at a time for it.

The bounds are what the routines need one after the other: ENERGY two
spectral and two PFF fields, ENEMON three, DIAGNOST seven, the right-hand
sides twelve (FORCE) and seven (NONLIN).  The half field
above a bound is for LN coefficients, tables and the allocator's granularity
(a field is 34 MB here)."""
import numpy as np
import pytest

import _oracle as O
from mlegs_amd import hip as H
from mlegs_amd.configs import CFG1
from test_gpu_parity import SMALL, Pair, relerr, state

pytestmark = pytest.mark.gpu

GRIDS = {
    "third": dict(nr=128, nth=128, nx=128, nrchop=85, ntchop=43, nxchop=43),
    "two_thirds": dict(nr=128, nth=128, nx=128, nrchop=85, ntchop=85, nxchop=43),
    "half_z": dict(nr=128, nth=128, nx=128, nrchop=85, ntchop=85, nxchop=64),
    "full": dict(nr=128, nth=128, nx=128, nrchop=122, ntchop=118, nxchop=64),
    "composite": dict(nr=120, nth=120, nx=130, nrchop=80, ntchop=40, nxchop=43),
}


def grown(cfg, call, nfields, before=None):
    import torch

    for _ in range(2):  # the first grid takes what the runtime keeps for the kernels
        g = H.Grid(dict(CFG1, **cfg))
        f = [g.scalar(H.FFF, np.zeros(g.shape(H.FFF), dtype=complex)) for _ in range(nfields)]
        if before:  # its band factors; it leaves one field with the pool
            before(f[0], f[1])
        g.synchronize()
        free = torch.cuda.mem_get_info()[0]
        call(*f)
        g.synchronize()
        n = (free - torch.cuda.mem_get_info()[0]) / (16.0 * np.prod(g.shape(H.PPP)))
        del f
        g.close()
    print(f"{n:.2f} fields")
    return n


@pytest.mark.parametrize("grid", list(GRIDS))
def test_buffers_of_the_diagnostics(grid):
    cfg = GRIDS[grid]
    assert grown(cfg, H.calc_boussi_energy, 3) <= 4.5
    assert grown(cfg, H.enemon, 2) <= 3.5
    assert grown(cfg, H.diagnost_it1, 2) <= 7.5


@pytest.mark.parametrize("grid", list(GRIDS))
def test_buffers_of_the_right_hand_sides(grid):
    cfg = GRIDS[grid]
    assert grown(cfg, H.calc_boussi_force, 6, H.idel2ln) <= 11.5
    assert grown(cfg, H.calc_boussi_nonlin, 8, H.idel2) <= 6.5


def test_right_hand_side_in_two_batches_and_in_place():
    """Truncations whose PFF fields take a buffer each, so that nine jobs go
    in two batches; results that are inputs give what separate ones do."""
    p = Pair(dict(SMALL, nr=24, nth=8, nx=8, nrchop=18, ntchop=8, nxchop=4))
    try:
        st = state(p)
        o, on = [p.o.field(O.FFF, a, ln) for a, ln in st], [p.o.field(O.FFF) for _ in range(3)]
        p.o.call("force", *o, *on)
        apart = None
        for same in ({}, {2: 2}, {0: 0, 1: 1, 2: 2}, {0: 1, 1: 2, 2: 0}):  # result -> the input that it is
            g = [p.g.scalar(O.FFF, a, ln) for a, ln in st]
            gn = [g[same[i]] if i in same else p.g.scalar(O.FFF) for i in range(3)]
            H.calc_boussi_force(*g, *gn)
            got = [x.download() for x in gn]
            if not same:
                apart = got
                for i in range(3):
                    p.check(gn[i], on[i], what=f"FORCE[{i}]")
            for x, y in zip(got, apart):
                assert np.array_equal(x[0], y[0]) and x[1:] == y[1:], same
    finally:
        p.close()


@pytest.mark.parametrize("cfg", [dict(SMALL, nr=24, nth=8, nx=8, nrchop=18, ntchop=8, nxchop=4),
                                 dict(SMALL, nr=24, nth=9, nx=6, nrchop=16, ntchop=6, nxchop=3),
                                 dict(SMALL, nth=12, nx=10, ntchop=7, nxchop=4)],
                         ids=["full", "two_thirds_half_z", "two_thirds"])
def test_diagnostics_at_wide_truncations(cfg):
    p = Pair(cfg)
    try:
        st = state(p, 1e-2)
        g = [p.g.scalar(O.FFF, a, ln) for a, ln in st]
        o = [p.o.field(O.FFF, a, ln) for a, ln in st]
        for a, b in zip(H.calc_boussi_energy(*g), p.o.energy(*o)):
            assert relerr(a, b) <= 1e-12
        p.g.chopset(3)
        O.lib().og_chopset(p.o.g, 3)
        for a, b in zip(H.enemon(*g[:2]), p.o.enemon(*o[:2])):
            assert relerr(a, b) <= 1e-12
        p.g.chopset(-3)
        O.lib().og_chopset(p.o.g, -3)
        d, ref = H.diagnost_it1(*g[:2]), dict(zip(H.DIAGNOST_IT1_KEYS, p.o.diagnost_it1(*o[:2])))
        # spreads and centre coordinates against what they are differences of
        size = dict(psiat1_spread=ref["psiat1"], chiat1_spread=ref["chiat1"], x=ref["r"], y=ref["r"])
        for k in H.DIAGNOST_IT1_KEYS:
            assert abs(d[k] - ref[k]) <= 1e-11 * max(abs(ref[k]), abs(size.get(k, 0.0))), k
    finally:
        p.close()
