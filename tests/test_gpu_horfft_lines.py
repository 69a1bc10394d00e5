"""The unscaled theta transforms of 16 .. 512 points against numpy, at the
sizes of both routes: fields within the 64 MB up to which the forward
transform goes on the line kernels, and past it; radial counts that end
inside a block of lines; truncations on both sides of 3/8 of NTH.  And
VDOTPSUB's padding, which its kernel writes.

Tolerance: as the mixed-radix transforms' (test_gpu_fft_any)."""
import numpy as np
import pytest

from mlegs_amd import hip as H
from mlegs_amd.configs import CFG1
from test_gpu_fft_any import rand, test_horfft as check, tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [16, 32, 64, 128, 256, 512])
@pytest.mark.parametrize("full", [False, True], ids=["third", "twothirds"])
def test_lines(n, full):
    check(n, full)


@pytest.mark.parametrize("n,nr,nx", [(64, 126, 480), (256, 62, 244), (512, 30, 250)])
def test_past_the_caches(n, nr, nx):
    ntc = n // 3
    g = H.Grid(dict(CFG1, nr=nr, nth=n, nx=nx, nrchop=12, ntchop=ntc, nxchop=1))
    try:
        assert 16 * np.prod(g.shape(H.PPP)) > 64e6
        x = np.zeros(g.shape(H.PFP), dtype=complex)
        x[:nr, :ntc] = rand((nr, ntc, nx), n)
        x[:, 0] = x[:, 0].real
        f = g.scalar(H.PFP, x)
        H.horfft(f, 1)
        got = f.e
        ref = np.fft.irfft(x[:nr, :ntc], n=2 * n, axis=1) * 2 * n
        ref = ref[:, 0::2] + 1j * ref[:, 1::2]
        assert np.max(np.abs(got[:nr, :n] - ref)) <= tol(n) * np.max(np.abs(ref))
        assert not got[nr:].any() and not got[:, n].any()
        H.horfft(f, -1)
        assert np.max(np.abs(f.e[:nr, :ntc] - x[:nr, :ntc])) <= 2 * tol(n) * np.max(np.abs(x)) * np.sqrt(n)
    finally:
        g.close()


@pytest.mark.parametrize("nr,nth,nx", [(12, 8, 6), (34, 9, 5)])
def test_vdotpsub_writes_its_padding(nr, nth, nx):
    g = H.Grid(dict(CFG1, nr=nr, nth=nth, nx=nx, nrchop=8, ntchop=3, nxchop=2))
    try:
        a = [rand(g.shape(H.PPP), i) for i in range(7)]
        f = [g.scalar(H.PPP, x) for x in a]
        r2 = np.asarray(g.table("r"))[:nr, None, None] ** 2
        H.vdotpsub(*f)
        a1, a2, a3, b1, b2, b3 = [x[:nr, :nth] for x in a[:6]]
        dot = lambda u, v: u.real * v.real + 1j * (u.imag * v.imag)
        ref = (dot(a1, b1) + dot(a2, b2)) / r2 + dot(a3, b3)
        got = f[6].e
        # three products, two sums, a quotient
        size = (np.abs(a1 * b1) + np.abs(a2 * b2)) / r2 + np.abs(a3 * b3)
        assert np.all(np.abs(got[:nr, :nth] - ref) <= 12 * 2.0 ** -53 * size)
        assert not got[nr:].any() and not got[:, nth:].any()
        # a result that is one of the inputs is cleared first
        H.vdotpsub(*f[:5], f[5], f[5])
        got = f[5].e
        ref = (dot(a1, b1) + dot(a2, b2)) / r2
        assert np.all(np.abs(got[:nr, :nth] - ref) <= 12 * 2.0 ** -53 * size)
    finally:
        g.close()
