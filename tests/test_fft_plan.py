"""The factorisation and digit reversal behind the any-length transforms
(mlegs_amd/csrc/fft_plan.h), compiled here and checked on the host: every
length from 2 to 4096 factors into radices with a butterfly and at most one
direct stage, the orders are permutations, and the in-place decimation in
frequency they describe is the DFT."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RADICES = {2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 16, 17, 19}
MAIN = r"""
#include <cstdio>
#include "fft_plan.h"
int main() {
  for (int n = 2; n <= 4096; n++) {
    mlg::FftFactors f;
    if (!mlg::fft_factor(n, f)) { std::printf("%d none\n", n); continue; }
    std::vector<int> freq, pos;
    mlg::fft_order(f, freq, pos);
    std::printf("%d %d %d", n, f.ns, f.direct);
    for (int i = 0; i < f.ns; i++) std::printf(" %d", f.rad[i]);
    for (int v : freq) std::printf(" %d", v);
    for (int v : pos) std::printf(" %d", v);
    std::printf("\n");
  }
}
"""


@pytest.fixture(scope="module")
def plans(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "main.cpp").write_text(MAIN)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "mlegs_amd", "csrc"), str(d / "main.cpp"),
                           "-o", str(d / "main")])
    out = {}
    for line in subprocess.check_output([str(d / "main")], text=True).splitlines():
        v = line.split()
        n, ns, direct = int(v[0]), int(v[1]), int(v[2])
        rad = [int(x) for x in v[3:3 + ns]]
        rest = np.array(v[3 + ns:], dtype=int)
        out[n] = (rad, direct, rest[:n // rad[-1]], rest[n // rad[-1]:])
    return out


FUSED = r"""
#include <cstdio>
#include "fft_plan.h"
int main() {
  for (int n = 2; n <= 4096; n++) {
    mlg::FusedPlan f;
    if (!mlg::fused_plan(n, f)) continue;
    std::printf("%d %d %d %d %d %ld %d", n, f.R, f.D, f.P, f.T, mlg::fused_lds(f), f.nmid);
    for (int i = 0; i < f.nmid; i++) std::printf(" %d", f.mid[i]);
    std::printf("\n");
  }
}
"""


def test_fused_plans_fit_their_block(tmp_path):
    (tmp_path / "main.cpp").write_text(FUSED)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "mlegs_amd", "csrc"),
                           str(tmp_path / "main.cpp"), "-o", str(tmp_path / "main")])
    got = {}
    for line in subprocess.check_output([str(tmp_path / "main")], text=True).splitlines():
        n, R, D, P, T, lds, nmid, *mid = [int(x) for x in line.split()]
        assert R * D * int(np.prod(mid, dtype=int)) == n and len(mid) == nmid and all(2 <= m <= 8 for m in mid) and 2 <= R <= 6
        assert D % 2 == 1 and D <= 61 and all(D % q for q in (3, 5, 7))
        assert T % 64 == 0 and n // R * P <= T <= 512 and 4 <= P <= 32
        lines = n * P * (1 + (D > 1))
        assert lines + n + n // 2 + 1 == lds and lds * 16 <= 160 * 1024
        assert (n // 2 + 1) <= (R // 2 + 1) * (T // P)
        got[n] = (R, D)
    for n in (3, 9, 12, 45, 90, 100, 122, 204, 306, 384, 512, 600, 640, 768):
        assert n in got, n
    assert not {289, 607, 608, 1000, 1024} & set(got)


def test_every_length_factors(plans):
    assert sorted(plans) == list(range(2, 4097))
    for n, (rad, direct, freq, pos) in plans.items():
        assert np.prod(rad) == n and len(rad) <= 8
        assert all(r in RADICES for r in (rad[:-1] if direct else rad))
        if direct:
            assert all(rad[-1] % p for p in (2, 3, 5, 7, 11, 13, 17, 19))
        assert len(freq) == n // rad[-1] and len(pos) == n
        assert np.array_equal(np.sort(pos), np.arange(n))
        f = (freq[:, None] + n // rad[-1] * np.arange(rad[-1])[None, :]).reshape(-1)  # frequency at each position
        assert np.array_equal(np.sort(f), np.arange(n)) and np.array_equal(pos[f], np.arange(n))


@pytest.mark.parametrize("n", [2, 17, 23, 46, 90, 204, 306, 384, 512, 529, 608, 1024, 3600])
def test_decimation_in_place_is_the_dft(plans, n):
    rad, _, freq, _ = plans[n]
    x = np.random.default_rng(n).standard_normal((2, n)).astype(complex)
    x = x[0] + 1j * x[1]
    s, L = x.copy(), n
    for R in rad:
        M = L // R
        w = np.exp(-2j * np.pi * np.outer(np.arange(R), np.arange(R)) / R)
        b = s.reshape(n // L, R, M)
        b = np.einsum("kq,bqj->bkj", w, b) * np.exp(-2j * np.pi * np.outer(np.arange(R), np.arange(M)) / L)
        s, L = b.reshape(-1), M
    y = np.empty(n, dtype=complex)
    R = rad[-1]
    y[(freq[:, None] + n // R * np.arange(R)[None, :]).reshape(-1)] = s
    assert np.max(np.abs(y - np.fft.fft(x))) <= 1e-12 * np.max(np.abs(y)) * np.log2(n)
