"""VERFFT and HORFFT at lengths of the mixed-radix kernels against numpy:
short lengths, summed directly (up to 24), a prime above 19 alone and with
factors (the direct stage), two to four stages, powers of two above 256, and
radial counts that leave part of a block's pencils empty.

Tolerance: an FFT of length N rounds within a few eps log2 N of the largest
value; the direct stage and the odd primes sum up to D terms (eps D / 2 at
most, D <= 4093 here, on values of unit size)."""
import numpy as np
import pytest

from mlegs_amd import hip as H
from mlegs_amd.configs import CFG1

pytestmark = pytest.mark.gpu

LENGTHS = [3, 5, 6, 7, 9, 10, 11, 12, 13, 15, 17, 19, 20, 21, 22, 23, 24, 25, 29, 46, 57, 90, 100, 143, 204, 289, 306, 384, 512, 529, 607, 608, 1024]


def tol(n):
    big = max(p for p in range(2, n + 1) if n % p == 0 and all(p % q for q in range(2, int(p ** 0.5) + 1)))
    return 2.0 ** -52 * (8 * np.log2(n) + big)


def rand(shape, seed):
    r = np.random.default_rng(seed)
    return r.standard_normal(shape) + 1j * r.standard_normal(shape)


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("full", [False, True], ids=["third", "half"])
def test_verfft(n, full):
    nxc = max(1, n // 2 if full else n // 3)
    cfg = dict(CFG1, nr=36, nth=4, nx=n, nrchop=12, ntchop=3, nxchop=nxc)
    g = H.Grid(cfg)
    try:
        a = np.zeros(g.shape(H.PFP), dtype=complex)
        a[:36, :3] = rand((36, 3, n), n)
        f = g.scalar(H.PFP, a)
        H.verfft(f, -1)
        ref = np.fft.fft(a[:, :3], axis=2) / n
        ref = np.concatenate([ref[:, :, :nxc], ref[:, :, n - nxc + 1:]], axis=2)
        got = f.e
        assert np.max(np.abs(got[:36] - ref[:36])) <= tol(n) * np.max(np.abs(ref)) * np.sqrt(n)
        b = np.zeros(g.shape(H.PFF), dtype=complex)
        b[:36] = rand((36, 3, 2 * nxc - 1), n + 1)
        f.upload(b, H.PFF)
        H.verfft(f, 1)
        z = np.zeros((39, 3, n), dtype=complex)
        z[:, :, :nxc] = b[:, :, :nxc]
        if nxc > 1:
            z[:, :, -(nxc - 1):] = b[:, :, nxc:]
        ref = np.fft.ifft(z, axis=2) * n
        assert np.max(np.abs(f.e[:, :3] - ref)) <= tol(n) * np.max(np.abs(ref))
    finally:
        g.close()


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("full", [False, True], ids=["third", "twothirds"])
def test_horfft(n, full):
    ntc = max(1, 2 * n // 3 if full else n // 3)
    cfg = dict(CFG1, nr=36, nth=n, nx=2, nrchop=12, ntchop=ntc, nxchop=1)
    g = H.Grid(cfg)
    try:
        v = np.random.default_rng(n).standard_normal((36, 2 * n, 2))
        a = np.zeros(g.shape(H.PPP), dtype=complex)
        a[:36, :n] = v[:, 0::2] + 1j * v[:, 1::2]
        f = g.scalar(H.PPP, a)
        H.horfft(f, -1)
        ref = np.fft.rfft(v, axis=1)[:, :ntc] / (2 * n)
        got = f.e
        assert np.max(np.abs(got[:36, :ntc] - ref)) <= tol(n) * np.max(np.abs(ref)) * np.sqrt(n)
        assert not got[36:, :ntc].any()
        x = np.zeros(g.shape(H.PFP), dtype=complex)
        x[:36, :ntc] = rand((36, ntc, 2), n + 1)
        x[:, 0] = x[:, 0].real
        f.upload(x, H.PFP)
        H.horfft(f, 1)
        ref = np.fft.irfft(x[:36, :ntc], n=2 * n, axis=1) * 2 * n
        got = f.e
        ref = ref[:, 0::2] + 1j * ref[:, 1::2]
        assert np.max(np.abs(got[:36, :n] - ref)) <= tol(n) * np.max(np.abs(ref))
        assert not got[36:].any() and not got[:, n].any()
    finally:
        g.close()


# two line buffers of 128 KB (a prime), one of 64 KB
@pytest.mark.parametrize("n", [4093, 4096])
def test_largest_lines(n):
    test_verfft(n, False)
    test_horfft(n, False)
