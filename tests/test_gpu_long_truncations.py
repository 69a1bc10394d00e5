"""The right-hand side at long truncations: the columns of its spectral
operators, six of them in one block, take 66 KB of LDS at NRCHOP 690 and 151
at 1600, near the end of the range (a block may have 160 KB; the normalised
functions of the reference's recurrence overflow between 1600 and 1700).

Tolerance: the largest change of the oracle's own results when its sums run
the other way (6e-12 of psi, 2e-11 of chi, 2e-15 of b), four times."""
import pytest

import _oracle as O
from mlegs_amd import hip as H
from test_gpu_parity import SMALL, TOL, Pair, relerr

pytestmark = pytest.mark.gpu


def oracle_force(p, st, reverse):
    O.lib().og_set_sum_order(reverse)
    try:
        o, on = [p.o.field(O.FFF, a, ln) for a, ln in st], [p.o.field(O.FFF) for _ in range(3)]
        p.o.call("force", *o, *on)
        return on
    finally:
        O.lib().og_set_sum_order(0)


@pytest.mark.parametrize("nrchop", [690, 1600])
def test_force(nrchop):
    p = Pair(dict(SMALL, nr=1730, nth=4, nx=2, nrchop=nrchop, ntchop=2, nxchop=1))
    try:
        st = [(p.noise(i, amp=0.1), ln) for i, ln in ((1, 0.5), (2, 0.0), (3, 0.0))]
        g, gn = [p.g.scalar(O.FFF, a, ln) for a, ln in st], [p.g.scalar(O.FFF) for _ in range(3)]
        H.calc_boussi_force(*g, *gn)
        for i, (a, b) in enumerate(zip(oracle_force(p, st, 0), oracle_force(p, st, 1))):
            p.check(gn[i], a, tol=max(TOL, 4 * relerr(b.arr(), a.arr())), what=f"FORCE[{i}]")
    finally:
        p.close()
