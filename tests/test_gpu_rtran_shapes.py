"""RTRAN backward against the oracle at sizes on both sides of the tile-shape
rule: node and column counts that a tile divides, one more and one fewer
(NR / 2 = 32, 33, 64, 65, 96; 2 NXCHOPDIM = 2, 30, 34, 62, 66, 98), few tiles
and more than three a CU.

Tolerance: the parity tests'."""
import pytest

import _oracle as O
from mlegs_amd import hip as H
from mlegs_amd.configs import CFG1
from test_gpu_parity import Pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr", [64, 66, 128, 130, 192])
@pytest.mark.parametrize("nxchop", [1, 8, 9, 16, 17, 25])
def test_rtran_backward(nr, nxchop):
    p = Pair(dict(CFG1, nr=nr, nth=32, nx=64, nrchop=nr - 20, ntchop=16, nxchop=nxchop))
    try:
        g, o = p.both(p.noise(1, 0), O.FFF, ln=0.37)
        H.rtran(g, 1)
        p.o.call("rtran", o, 1)
        p.check(g, o, what="RTRAN backward")
    finally:
        p.close()


@pytest.mark.parametrize("nr,nxchop", [(66, 43), (128, 43), (130, 64)])
def test_many_tiles(nr, nxchop):
    p = Pair(dict(CFG1, nr=nr, nth=512, nx=128, nrchop=nr - 2, ntchop=nr - 8, nxchop=nxchop))
    try:
        g, o = p.both(p.noise(1, 0), O.FFF, ln=0.37)
        H.rtran(g, 1)
        p.o.call("rtran", o, 1)
        p.check(g, o, what="RTRAN backward")
    finally:
        p.close()
