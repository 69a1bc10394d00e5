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

}  // namespace mlg
