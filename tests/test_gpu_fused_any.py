"""The fused products (FORCE with its linear terms, NONLIN without) at theta
lengths of k_fused_any against the FP64 oracle: every radix of the last stage
(6, 5, 4, 3, 2), middle stages, a direct stage (factors 11 .. 61), both
truncations in use (a third and two thirds of NTH), radial counts that leave
part of a block empty; and lengths without a plan (49, 289, 608), which take
the separate transforms.

Tolerance: the parity tests' 1e-12, ten times that for chi (the inverse
Laplacian's conditioning)."""
import pytest

import _oracle as O
from mlegs_amd import hip as H
from mlegs_amd.configs import CFG1
from test_gpu_parity import TOL, Pair, state

pytestmark = pytest.mark.gpu

LENGTHS = [2, 3, 4, 5, 6, 7, 8, 9, 10, 12, 14, 16, 20, 22, 32, 45, 49, 66, 81, 90, 100, 104, 126, 153, 204, 289, 306, 310, 366, 384, 512, 608, 640, 768]


@pytest.mark.parametrize("nth", LENGTHS)
@pytest.mark.parametrize("full", [False, True], ids=["third", "twothirds"])
def test_right_hand_sides(nth, full):
    ntc = min(max(1, 2 * nth // 3 if full else nth // 3 + 1), nth)
    nr, nrchop = (36, 24) if nth < 100 else (12, 8)
    compare(dict(CFG1, nr=nr, nth=nth, nx=6, nrchop=nrchop, ntchop=ntc, nxchop=3))


# more than 768 blocks of a wave a field (64, 32, .. 1 of the 15 lines of a plane each), more than 4096 at 512
@pytest.mark.parametrize("nth,nx", [(8, 800), (16, 800), (32, 800), (64, 400), (128, 200), (256, 100), (512, 54),
                                    (512, 280)])
@pytest.mark.parametrize("full", [False, True], ids=["third", "twothirds"])
def test_right_hand_sides_on_large_grids(nth, nx, full):
    ntc = 2 * nth // 3 if full else nth // 3
    compare(dict(CFG1, nr=12, nth=nth, nx=nx, nrchop=8, ntchop=ntc, nxchop=3))


def compare(cfg):
    p = Pair(cfg)
    try:
        st = state(p, 1e-3)
        outs = [p.empty() for _ in range(3)]
        ins = [p.both(a, O.FFF, ln) for a, ln in st]
        H.calc_boussi_force(*[x[0] for x in ins], *[x[0] for x in outs])
        p.o.call("force", *[x[1] for x in ins], *[x[1] for x in outs])
        for (g, o), nm in zip(outs, ("psin", "chin", "bn")):
            p.check(g, o, tol=TOL if nm != "chin" else 10 * TOL, what=nm)
        v = [p.empty() for _ in range(7)]
        p.g.chopset(3)
        p.o.chopset(3)
        H.pc2vel(ins[0][0], ins[1][0], *[x[0] for x in v[:3]])
        H.pc2vor(ins[0][0], ins[1][0], *[x[0] for x in v[3:6]])
        p.o.call("pc2vel", ins[0][1], ins[1][1], *[x[1] for x in v[:3]])
        p.o.call("pc2vor", ins[0][1], ins[1][1], *[x[1] for x in v[3:6]])
        p.g.chopset(-3)
        p.o.chopset(-3)
        H.calc_boussi_nonlin(ins[2][0], *[x[0] for x in v[:3]], v[6][0], *[x[0] for x in v[3:6]])
        p.o.call("nonlin", ins[2][1], *[x[1] for x in v[:3]], v[6][1], *[x[1] for x in v[3:6]])
        for (g, o), nm in zip(v, ("rur", "rup", "uz", "ror", "rop", "oz", "bn")):
            p.check(g, o, tol=10 * TOL if nm in ("ror", "rop", "oz") else TOL, what=nm)
    finally:
        p.close()
