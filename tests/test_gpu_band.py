"""GPU vs oracle: the banded solves of IDEL2, IDEL2LN and IHELM
(src/mod_legops.f90:823-1354 on LUDCMPB/LUBKSBB, src/mod_bandmat.f90:
65-156,320-402) on both of the library's routes, and AB2-CN / ETD2 steps
there (the viscous step's three solves share one launch).  From NRCHOP 20 to
512 every penta-diagonal system runs on several lanes, 8 rows each (NRCHOP 20:
4 lanes, 48 and 64: 8, 96 and 128: 16, 200 and 256: 32, 512: 64); below 20
and above 512 one thread runs each system, by LUBKSBB's arithmetic (below 20,
AB2-CN steps with diffusion of all fields take the lanes)."""
import pytest

import _oracle as O
from mlegs_amd import hip as H
from mlegs_amd.configs import CFG1
from test_gpu_parity import SMALL_ETD, Pair, run_steps

pytestmark = pytest.mark.gpu

GRIDS = {
    "nrchop12": dict(CFG1, nr=24, nth=16, nx=16, nrchop=12, ntchop=6, nxchop=5),
    "nrchop19": dict(CFG1, nr=32, nth=16, nx=16, nrchop=19, ntchop=6, nxchop=5),
    "nrchop20": dict(CFG1, nr=32, nth=16, nx=16, nrchop=20, ntchop=6, nxchop=5),
    "nrchop48": dict(CFG1, nr=64, nth=16, nx=16, nrchop=48, ntchop=6, nxchop=5),
    "nrchop64": dict(CFG1, nr=96, nth=16, nx=16, nrchop=64, ntchop=6, nxchop=5),
    "nrchop96": dict(CFG1, nr=128, nth=16, nx=16, nrchop=96, ntchop=6, nxchop=5),
    "nrchop128": dict(CFG1, nr=192, nth=16, nx=16, nrchop=128, ntchop=6, nxchop=5),
    "nrchop200": dict(CFG1, nr=300, nth=16, nx=16, nrchop=200, ntchop=6, nxchop=5),
    "nrchop256": dict(CFG1, nr=384, nth=16, nx=16, nrchop=256, ntchop=6, nxchop=5),
    "nrchop512": dict(CFG1, nr=768, nth=16, nx=16, nrchop=512, ntchop=6, nxchop=5),
    "nrchop520": dict(CFG1, nr=780, nth=16, nx=16, nrchop=520, ntchop=6, nxchop=5),
}
TOL = 1e-12


def bar(cfg, case):
    """IDEL2LN's inverse grows ill-conditioned as NRCHOP^2: the oracle's own
    result moves by 4e-15, 2e-14, 4e-14 and 2.4e-13 (relative) at NRCHOP 64,
    128, 256 and 512 when its right-hand side is perturbed by one ulp, and a
    solve that rounds differently (the partitioned substitution carries its
    segment states) differs from it by 3e-14 .. 2.2e-12 over the same range.
    Its bar is 1e-12 at NRCHOP 181 and grows as NRCHOP^2 above that."""
    if case != "idel2ln":
        return TOL
    return TOL * max(1.0, 2.0 * (cfg["nrchop"] / 256.0) ** 2)


@pytest.fixture(scope="module", params=list(GRIDS))
def P(request):
    p = Pair(GRIDS[request.param])
    yield p
    p.close()


@pytest.mark.parametrize("case", ["idel2", "idel2_ln", "idel2ln", "ihelm"])
def test_solves_match_oracle(P, case):
    gb, ob = P.both(P.noise(4), O.FFF, ln=0.6)
    ga, oa = P.empty()
    if case == "idel2":
        H.idel2(gb, ga)
        P.o.call("idel2", ob, oa, 0, 0.0)
    elif case == "idel2_ln":
        H.idel2(gb, ga, ln=-0.8)
        P.o.call("idel2", ob, oa, 1, -0.8)
    elif case == "idel2ln":
        H.idel2ln(gb, ga)
        P.o.call("idel2ln", ob, oa)
    else:
        H.ihelm(gb, ga, 2.0 / 1e-3 / 1e-3)
        P.o.call("ihelm", ob, oa, 2.0 / 1e-3 / 1e-3)
    e = P.check(ga, oa, tol=bar(P.cfg, case), what=case)
    print(f"{case}: rel err {e:.2e}")
    if not 20 <= P.cfg["nrchop"] <= 512:
        assert e == 0.0, "LUBKSBB's arithmetic"


@pytest.mark.parametrize("grid", ["nrchop12", "nrchop19", "nrchop128", "nrchop520"])
def test_ab2_cn_steps(grid):
    run_steps(GRIDS[grid], 3)


@pytest.mark.parametrize("grid", ["nrchop19", "nrchop200", "nrchop520"])
def test_etd2_steps(grid):
    cfg = dict(GRIDS[grid], **{k: SMALL_ETD[k] for k in ("adams", "hyper_cn", "nup", "kappap", "visc_p", "omega", "bv0")})
    run_steps(cfg, 3)
