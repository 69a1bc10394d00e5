"""DIAGNOST's every-IT1 section against the oracle at sizes where the sums over
the physical grid have remainders: radial nodes past a block of 64, planes
that four ranges of z do not divide, odd theta lengths; same tolerance and
scales as the other sizes."""
import pytest

from test_gpu_diagnost import test_diagnost_it1_matches_oracle as check
from test_gpu_parity import SMALL

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nr,nth,nx", [(16, 8, 2), (64, 8, 4), (66, 12, 6), (130, 9, 5), (62, 90, 10)])
def test_sums_over_the_physical_grid(nr, nth, nx):
    check(dict(SMALL, nr=nr, nth=nth, nx=nx, nrchop=nr - 8, ntchop=3, nxchop=min(2, nx // 2)))
