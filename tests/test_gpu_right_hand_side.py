"""The AB2-CN right-hand side and viscous step in their fused launches, and
the band solves at short truncations, against the FP64 oracle.

* CALC_BOUSSI_FORCE with b (and psi, chi) holding rows past NRCHOP: GRAD sees
  them (NRCHOP+3), W = TOFP(COPY0 b) does not.
* The AB2 step formed with VISC2's right-hand sides: a start state with rows
  past the truncation is chopped by it, kappa = 0 (b not diffused) and
  VISC%SW = 0 take the separate launches.
* Band solves at NRCHOP 4 .. 63 on 2, 4 and 8 lanes a system (edges of the
  8-row segments), and their transposes.

Tolerances are those of the parity tests: 1e-12 for one routine; steps
max(1e-12, 6 s), s the oracle's own change under reversed Legendre sums."""
import numpy as np
import pytest

import _oracle as O
from mlegs_amd import hip as H
from mlegs_amd.configs import CFG1
from test_gpu_parity import TOL, Pair, relerr, run_steps

pytestmark = pytest.mark.gpu

BASE = dict(CFG1, nr=40, nth=16, nx=12, nrchop=26, ntchop=6, nxchop=5)


@pytest.mark.parametrize("cfg", [BASE, dict(BASE, nth=64, ntchop=22), dict(BASE, nx=18, nxchop=9), dict(BASE, nth=32, nx=8, ntchop=21, nxchop=3)],
                         ids=["16x12", "64x12", "16x18", "32x8full"])
def test_force_sees_rows_past_nrchop(cfg):
    p = Pair(cfg)
    try:
        ins = [p.both(p.noise(i + 1, iof=3), O.FFF, ln=0.4 if i == 0 else 0.0) for i in range(3)]
        # DEL2's check: chi's top m = 1 row at NRCHOP+3 must vanish
        chi = ins[1][0].e.copy(order="F")
        chi[cfg["nrchop"] + 1, 1, :] = 0
        ins[1] = p.both(chi, O.FFF)
        outs = [p.empty() for _ in range(3)]
        H.calc_boussi_force(*[x[0] for x in ins], *[x[0] for x in outs])
        p.o.call("force", *[x[1] for x in ins], *[x[1] for x in outs])
        for (g, o), nm in zip(outs, ("psin", "chin", "bn")):
            # chin: the inverse Laplacian's conditioning (its LN row cancels)
            p.check(g, o, tol=TOL if nm != "chin" else 10 * TOL, what=nm)
    finally:
        p.close()


def test_ab2_step_chops_a_start_state():
    p = Pair(BASE)
    try:
        st = [p.noise(i + 1, iof=2, amp=1e-4) for i in range(3)]
        st[1][BASE["nrchop"]:, 1, :] = 0
        g = [p.g.scalar(O.FFF, a) for a in st]
        o = [p.o.field(O.FFF, a) for a in st]
        gs, osv = H.Solver(p.g), O.OSolver(p.o)
        gs.time_step(*g)  # no start: the history is zero on both sides
        assert osv.step(*o) == 0
        for a, b, nm in zip(g, o, ("psi", "chi", "b")):
            x, y = a.e, b.arr()
            assert relerr(x, y) <= 10 * TOL, nm
            for m in range(BASE["ntchop"]):
                assert not x[BASE["nrchop"] - m:, m, :].any(), nm
        gs.close()
        osv.close()
    finally:
        p.close()


@pytest.mark.parametrize("change", [dict(kappa=0.0), dict(visc_sw=0), dict(nrchop=33, nr=48), dict(nr=80, nrchop=63)],
                         ids=["kappa0", "inviscid", "nrchop33", "nrchop63"])
def test_ab2_steps(change):
    run_steps(dict(BASE, **change), 3)


@pytest.mark.parametrize("nrchop", [4, 7, 8, 9, 16, 17, 31, 32, 33, 48, 63])
def test_short_band_solves(nrchop):
    cfg = dict(CFG1, nr=2 * nrchop + 8, nth=16, nx=16, nrchop=nrchop, ntchop=min(6, nrchop - 1), nxchop=5)
    p = Pair(cfg)
    try:
        for case in ("idel2", "idel2_ln", "idel2ln", "ihelm"):
            gb, ob = p.both(p.noise(4), O.FFF, ln=0.6)
            ga, oa = p.empty()
            if case.startswith("idel2") and case != "idel2ln":
                ln = None if case == "idel2" else -0.8
                H.idel2(gb, ga, ln=ln)
                p.o.call("idel2", ob, oa, 0 if ln is None else 1, 0.0 if ln is None else ln)
            elif case == "idel2ln":
                H.idel2ln(gb, ga)
                p.o.call("idel2ln", ob, oa)
            else:
                H.ihelm(gb, ga, 2.0 / 1e-3 / 1e-3)
                p.o.call("ihelm", ob, oa, 2.0 / 1e-3 / 1e-3)
            p.check(ga, oa, what=f"{case} at {nrchop}")
        # <A^-T y, x> = <y, A^-1 x> for IHELM, with its log term
        rng = np.random.default_rng(nrchop)
        x, y = [p.rand(O.FFF, int(rng.integers(1 << 30))) for _ in range(2)]
        keep = np.zeros(x.shape)
        for m in range(cfg["ntchop"]):
            keep[:nrchop - m, m, :] = 1
        x, y = np.asfortranarray(x * keep), np.asfortranarray(y * keep)
        fx, fy, sx, sy = p.g.scalar(O.FFF, x, 0.3), p.g.scalar(O.FFF, y, -0.2), p.g.scalar(), p.g.scalar()
        H.ihelm(fx, sx, 1e3)
        H.adjoint_op(H.ADJ_IHELM, [fy, sy], 1e3)
        a = np.sum((np.conj(y) * sx.e).real) + -0.2 * sx.ln
        b = np.sum((np.conj(sy.e) * x).real) + 0.3 * sy.ln
        assert abs(a - b) <= 1e-12 * np.linalg.norm(y) * np.linalg.norm(sx.e)
    finally:
        p.close()
