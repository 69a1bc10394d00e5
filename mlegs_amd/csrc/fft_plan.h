// Factorisation of a transform length for the mixed-radix FFT kernels
// (k_fft_any.hip).  Host code only: no HIP types.
#pragma once
#include <vector>

namespace mlg {

// Radices with a butterfly in registers.  A prime factor above 19 has none:
// the product of all such factors is the length of a last, direct stage.
constexpr int FFT_RADICES[] = {2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 16, 17, 19};
constexpr int FFT_MAX_STAGES = 8;

struct FftFactors {
  int n = 0;
  int ns = 0;                      // stages, the direct one included
  int rad[FFT_MAX_STAGES] = {0};   // radix of each stage, in order
  int direct = 0;                  // 1: the last stage sums directly
};

// The fewest stages whose radices multiply to n, and among those the smallest
// sum of radices; best, cur: stage lists, largest radix first.
inline void fft_search(int n, int maxr, std::vector<int> &cur, std::vector<int> &best) {
  if (n == 1) {
    auto sum = [](const std::vector<int> &v) {
      int s = 0;
      for (int x : v) s += x;
      return s;
    };
    if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && sum(cur) < sum(best))) best = cur;
    return;
  }
  if (!best.empty() && cur.size() >= best.size()) return;
  for (int i = (int)(sizeof(FFT_RADICES) / sizeof(int)) - 1; i >= 0; i--) {
    const int r = FFT_RADICES[i];
    if (r > maxr || n % r) continue;
    cur.push_back(r);
    fft_search(n / r, r, cur, best);
    cur.pop_back();
  }
}

// n >= 2.  Returns false if n has no factorisation within FFT_MAX_STAGES.
inline bool fft_factor(int n, FftFactors &f) {
  int smooth = n, direct = 1;
  for (int p = 2; p <= 19; p++)
    while (smooth % p == 0 && (p == 2 || p == 3 || p == 5 || p == 7 || p == 11 || p == 13 || p == 17 || p == 19)) {
      smooth /= p;
      direct *= p;
    }
  // smooth now holds the factors above 19, direct the rest
  const int big = smooth, rest = direct;
  std::vector<int> cur, best;
  if (rest > 1) fft_search(rest, 19, cur, best);
  f = FftFactors{};
  f.n = n;
  f.ns = (int)best.size() + (big > 1 ? 1 : 0);
  f.direct = big > 1;
  if (f.ns < 1 || f.ns > FFT_MAX_STAGES) return false;
  for (size_t i = 0; i < best.size(); i++) f.rad[i] = best[i];
  if (big > 1) f.rad[f.ns - 1] = big;
  return true;
}

// Decimation in frequency in place: block b of the last stage (radix R)
// holds the outputs of frequencies freq[b] + (n / R) k, k < R, at positions
// b R + k.  freq has n / R entries; pos[frequency] = position, n entries.
inline void fft_order(const FftFactors &f, std::vector<int> &freq, std::vector<int> &pos) {
  const int R = f.rad[f.ns - 1], nb = f.n / R;
  freq.assign(nb, 0);
  pos.assign(f.n, 0);
  for (int b = 0; b < nb; b++) {
    // digits of b, first stage most significant, become those of the
    // frequency, first stage least significant
    int rest = b, size = nb, place = 1, k = 0;
    for (int s = 0; s + 1 < f.ns; s++) {
      size /= f.rad[s];
      k += (rest / size) * place;
      rest %= size;
      place *= f.rad[s];
    }
    freq[b] = k;
    for (int q = 0; q < R; q++) pos[k + nb * q] = b * R + q;
  }
}

// The fused products at a theta length n (k_fused_any.hip): the line's last
// inverse stage has radix R = 2..6 and leaves each thread R physical points;
// before it come middle stages of radix 2..8 and, first, a direct stage over
// the product D of the prime factors above 7.
struct FusedPlan {
  int n = 0;                         // 0: not planned
  int R = 0, D = 1, nmid = 0;        // n = D mid[0] .. mid[nmid-1] R
  int mid[FFT_MAX_STAGES] = {0};
  int P = 0, T = 0;                  // radial lines and threads of a block
};
// LDS of a block in 16-byte values: the roots, one line buffer, and a second
// one for the direct stage
inline long fused_lds(const FusedPlan &f) {
  return f.n + f.n / 2 + 1 + (long)f.n * f.P * (1 + (f.D > 1));
}
inline bool fused_plan(int n, FusedPlan &f) {
  f = FusedPlan{};
  int rest = n, D = 1;
  for (int p : {2, 3, 5, 7})
    while (rest % p == 0) rest /= p;
  D = rest;
  // a direct stage reads D / 2 values for each one it forms; at NR = 192, NX =
  // 64 the kernel takes 426 us for NTH = 122 (D = 61) where the separate
  // transforms and products take 601; no configured length has a larger one
  if (D > 61) return false;
  // six or five points a thread in blocks of four waves are the fastest (FORCE
  // kernel at NTH = 204, NR = 408, NX = 128: 1.45 ms against 1.56 with four
  // points in eight waves; NTH = 384, NX = 64: 0.81 against 1.21).  Seven and
  // eight (NTH = 384: 1.30 ms) are slowed by their registers, and lengths that
  // only they would take stay with the separate kernels (NTH = 608, NR = 64,
  // NX = 64: 750 us with eight points, 688 apart)
  for (int R : {6, 5, 4, 3, 2}) {
    if (n % (D * R)) continue;
    FusedPlan c;
    c.n = n;
    c.R = R;
    c.D = D;
    std::vector<int> cur, best;
    const int m = n / (D * R);
    if (m > 1) {
      fft_search(m, 8, cur, best);
      if (best.empty()) continue;
    }
    c.nmid = (int)best.size();
    if (c.nmid + 2 > FFT_MAX_STAGES) continue;
    for (int i = 0; i < c.nmid; i++) c.mid[i] = best[i];
    c.P = (R == 5 || R == 6 ? 256 : 512) * R / n;
    if (c.P < 4) c.P = 512 * R / n;
    if (c.P > 32) c.P = 32;
    while (c.P > 0 && fused_lds(c) * 16 > 156 * 1024) c.P--;
    if (c.P < 4) continue;  // shorter runs of r than 64 bytes
    c.T = (n / R * c.P + 63) / 64 * 64;
    // the line's n / 2 + 1 pairs, R / 2 + 1 a thread
    if ((n / 2 + 1) > (R / 2 + 1) * (c.T / c.P)) continue;
    f = c;
    return true;
  }
  return false;
}
}  // namespace mlg
