"""The transposed operators at the lengths and truncations whose kernels
test_gpu_adjoint's 32x16x16 grid does not reach: the scaled theta transforms
(m = 0 and m >= 1 differently, with the Gauss weights on TOFF's way) as short
sums, mixed radices, direct stages and at 512 points, and the transposed band
solves on one thread a system below NRCHOP 20 and above 512.

The tolerances are relative to the sizes of the factors (check_dot).  The
solves' is the one of the solves themselves (test_gpu_band); a step's two
sides go through all of these and a central difference of states of unit size
against directions of 1e-2."""
import pytest

import test_gpu_adjoint as T
from mlegs_amd import adjoint as A
from mlegs_amd import hip as H

pytestmark = pytest.mark.gpu

LENGTHS = {
    "theta12_z12": dict(nth=12, nx=12, ntchop=5, nxchop=4),
    "theta15_z30": dict(nth=15, nx=30, ntchop=6, nxchop=10),
    "theta30_z46": dict(nth=30, nx=46, ntchop=10, nxchop=15),
    "theta46_z9": dict(nth=46, nx=9, ntchop=16, nxchop=3),
    "theta29_full": dict(nth=29, nx=16, ntchop=18, nxchop=8),
    "theta512": dict(nth=512, nx=8, ntchop=18, nxchop=3),
}
TRUNCATIONS = {
    "nrchop14": dict(nr=24, nrchop=14),
    "nrchop19": dict(nr=30, nrchop=19),
    "nrchop48": dict(nr=72, nrchop=48),
    "nrchop520": dict(nr=780, nrchop=520, nth=8, nx=4, ntchop=3, nxchop=2),
}


def march(cfg):
    import torch

    torch.cuda.set_device(0)
    m = A.March(H.Grid(cfg))
    m.cfg = cfg
    return m


@pytest.fixture(params=list(LENGTHS))
def L(request):
    m = march(dict(T.SMALL_AB, **LENGTHS[request.param]))
    yield m
    m.close()
    m.grid.close()


def test_transposed_transforms(L):
    T.test_transposed_transforms(L)


def test_transposed_project(L):
    T.test_transposed_project(L)


def test_step_adjoint(L):
    x, d, ybar = T.state(L, 1e-2), T.direction(L, 31, 1e-2), T.direction(L, 41, 1.0)
    eps = 0.5
    lin = (L.step(x + eps * d, False) - L.step(x - eps * d, False)) / (2 * eps)
    xbar = L.step_adjoint(x, ybar, False)
    T.check_dot(T.dot(lin, ybar), T.dot(d, xbar), "STEP_BOUSSI_AB_CN")


@pytest.mark.parametrize("name", list(TRUNCATIONS))
def test_transposed_solves(name):
    cfg = dict(T.SMALL_AB, **TRUNCATIONS[name])
    g = H.Grid(cfg)
    tol = 1e-12 * max(1.0, 2.0 * (cfg["nrchop"] / 256.0) ** 2)
    alp, ln = 2 / cfg["nu"] / cfg["dt"], 0.37
    for op, what in ((H.ADJ_IDEL2LN, "IDEL2LN"), (H.ADJ_IHELM, "IHELM")):
        b, ab = T.fff(g, cfg, 30), T.fff(g, cfg, 31)
        bln = 0.0 if op == H.ADJ_IDEL2LN else -0.21
        gb, ga = g.scalar(H.FFF, b, bln), g.scalar()
        if op == H.ADJ_IDEL2LN:
            H.idel2ln(gb, ga)
        else:
            H.ihelm(gb, ga, alp)
        a, _, aln = ga.download()
        f = [g.scalar(H.FFF, ab, ln), g.scalar()]
        H.adjoint_op(op, f, alp)
        bb, _, bbln = f[1].download()
        size = T.sizes((a, ab), (b, bb)) + abs(aln * ln) + abs(bln * bbln)
        T.check_dot(T.fdot(a, ab) + aln * ln, T.fdot(b, bb) + bln * bbln, what, size, tol)
        del gb, ga, f
    g.close()
