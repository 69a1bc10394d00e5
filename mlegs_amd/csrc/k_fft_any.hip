// Axial (z) and azimuthal (theta) transforms of any length: mixed-radix FFTs
// over radial pencils, for the lengths the four-step register kernels of
// k_fft.hip do not take (not a power of two, or above 256).  The reference
// plans FFTW at any length (src/mod_fft.f90:833-920,1006-1091).
//
// One block owns P consecutive radial nodes of one (m, field) or z plane and
// transforms their lines in LDS, [position][pencil] with the pencils fastest,
// so that global accesses are runs of P consecutive r and LDS accesses are
// free of bank conflicts.  Decimation in frequency in place: stage s of
// radix R on blocks of length L reads x[j + (L/R) q], does an R-point DFT in
// registers, multiplies by W_L^{jk} and writes the same positions back, so a
// stage needs one barrier and no second buffer.  The first stage loads from
// global memory and the last one stores to it; the digit-reversed order of
// the results costs nothing there, a line's every element being its own run
// of r.  Bound: HBM (16 B in and out per element); LDS is passed stages - 1
// times.  A prime factor above 19 is summed directly in the last stage.
//
// Direct O(N^2) sums, and radix-2 stages in LDS for powers of two above 256,
// took these lengths before (up to 24 points direct sums still do).  Per field at NTH = 204, NX = 608 (NR = 408, 136
// modes, 607 wavenumbers; 1.09 GB a z-transform, 1.36 GB a theta transform):
//   VERFFT backward 11.0 -> 0.36 ms, forward 13.5 -> 0.37 (3.0 TB/s)
//   HORFFT backward  6.5 -> 0.65 ms, forward  7.4 -> 0.44 (2.1, 3.1 TB/s)
// and at NTH = 512, NX = 384 (NR = 192): 1.84 -> 0.14, 3.13 -> 0.13, 0.76 ->
// 0.40 and 0.73 -> 0.30 ms.
#include "fft_radix.h"
#include "mlegs_internal.h"
#include "xcd.h"

namespace mlg {

// rounds like any FFT, not operation for operation like a reference library
#pragma clang fp contract(fast)

namespace {

using namespace fftr;

// One stage: blocks of length L; i0, istep: the thread's first butterfly and
// the stride to its next one.  ld(position) -> value; st(position, block,
// output, value).
template <int R, bool INV, class LD, class ST>
__device__ __forceinline__ void stage(int n, int L, int i0, int istep, const double2 *__restrict__ tw, LD ld, ST st) {
  const int M = L / R, nb = n / R, step = n / L;
  for (int i = i0; i < nb; i += istep) {
    const int b = i / M, j = i - b * M, base = b * L + j;
    double2 v[R];
#pragma unroll
    for (int q = 0; q < R; q++) v[q] = ld(base + M * q);
    Dft<R, INV>::run(v, tw, nb);
    if (M > 1) {
#pragma unroll
      for (int k = 1; k < R; k++) v[k] = rmul<INV>(v[k], tw[j * k * step]);
    }
#pragma unroll
    for (int k = 0; k < R; k++) st(base + M * k, b, k, v[k]);
  }
}

#define FFT_ANY_RADIX(R_, CALL) \
  switch (R_) {                 \
    case 2: CALL(2); break;     \
    case 3: CALL(3); break;     \
    case 4: CALL(4); break;     \
    case 5: CALL(5); break;     \
    case 6: CALL(6); break;     \
    case 7: CALL(7); break;     \
    case 8: CALL(8); break;     \
    case 9: CALL(9); break;     \
    case 10: CALL(10); break;   \
    case 11: CALL(11); break;   \
    case 12: CALL(12); break;   \
    case 13: CALL(13); break;   \
    case 16: CALL(16); break;   \
    case 17: CALL(17); break;   \
    case 19: CALL(19); break;   \
    default: break;             \
  }

// The direct last stage of length D (odd, every prime factor above 19):
// outputs k and D - k of block b together.  in: the staged positions.
template <bool INV, class ST>
__device__ __forceinline__ void stage_direct(int n, int D, int i0, int istep, const double2 *__restrict__ tw,
                                             const double2 *s, int P, int p, ST st) {
  const int H = (D - 1) / 2, step = n / D, items = step * (H + 1);
  for (int i = i0; i < items; i += istep) {
    const int b = i / (H + 1), k = i - b * (H + 1);
    const double2 *x = s + (size_t)b * D * P + p;
    double2 A = x[0], B = make_double2(0.0, 0.0);
    int ph = 0;
    for (int q = 1; q <= H; q++) {
      const double2 u = x[q * P], w = x[(D - q) * P];
      ph += k;
      if (ph >= D) ph -= D;
      const double2 t = tw[ph * step];
      A.x += (u.x + w.x) * t.x;
      A.y += (u.y + w.y) * t.x;
      B.x += (u.x - w.x) * t.y;
      B.y += (u.y - w.y) * t.y;
    }
    const double2 jb = INV ? make_double2(B.y, -B.x) : make_double2(-B.y, B.x);
    st(b * D + k, b, k, cadd(A, jb));
    if (k > 0) st(b * D + D - k, b, D - k, csub(A, jb));
  }
}

}  // namespace

// All stages of the block's lines.  ld(position) loads an input of the
// thread's pencil, st(position, frequency, value) takes the results.  s:
// LDS, [position][pencil]; STAGED: the inputs lie there already (ld is not
// called).  Every thread of the block calls it.
template <bool INV, bool STAGED = false, class LD, class ST>
__device__ __forceinline__ void fft_any(const FftAny &f, const double2 *__restrict__ tw, double2 *s, int lgp, LD ld, ST st) {
  const int P = 1 << lgp, p = threadIdx.x & (P - 1), i0 = threadIdx.x >> lgp, istep = blockDim.x >> lgp;
  const int n = f.n, last = f.ns - 1;
  auto lds_ld = [&](int pos) { return s[(pos << lgp) + p]; };
  auto lds_st = [&](int pos, int, int, double2 v) { s[(pos << lgp) + p] = v; };
  const int outstep = n / f.rad[last];
  auto out = [&](int pos, int b, int k, double2 v) { st(pos, f.freq[b] + outstep * k, v); };
  int L = n, q = 0;
  if (!STAGED) {
    if (last == 0) {  // direct only (lengths of one butterfly are summed, fft_short): stage the line as it lies
      for (int i = i0; i < n; i += istep) s[(i << lgp) + p] = ld(i);
    } else {
#define C_FIRST(R_) stage<R_, INV>(n, n, i0, istep, tw, ld, lds_st)
      FFT_ANY_RADIX(f.rad[0], C_FIRST)
#undef C_FIRST
      L /= f.rad[0];
      q = 1;
    }
    __syncthreads();
  }
  for (; q < last; q++) {
#define C_MID(R_) stage<R_, INV>(n, L, i0, istep, tw, lds_ld, lds_st)
    FFT_ANY_RADIX(f.rad[q], C_MID)
#undef C_MID
    __syncthreads();
    L /= f.rad[q];
  }
  if (f.direct) {
    stage_direct<INV>(n, L, i0, istep, tw, s, P, p, out);
  } else {
#define C_LAST(R_) stage<R_, INV>(n, L, i0, istep, tw, lds_ld, out)
    FFT_ANY_RADIX(f.rad[last], C_LAST)
#undef C_LAST
  }
}

// ---- VERFFT forward: PFP (r, m, z) -> PFF (r, m, k), / NX.  Logical block:
// radial chunk fastest, then mode, then field, grouped per XCD: neighbouring
// chunks share the lines that a run of P nodes straddles.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_verfft_fwd_any(KGrid g, FftAny f, int lgp, const double2 *__restrict__ tw, TransformJobs jobs, int nj) {
  extern __shared__ double2 s[];
  const int P = 1 << lgp, nrb = (g.ndimr + P - 1) >> lgp;
  const int lid = xcd_logical(nrb * g.ntchopdim * nj);
  if (lid < 0) return;
  const int bx = lid % nrb, rest = lid / nrb, mm = rest % g.ntchopdim, fj = rest / g.ntchopdim;
  const int rr = (bx << lgp) + (threadIdx.x & (P - 1));
  const bool live = rr < g.nr, inr = rr < g.ndimr;
  const double2 *__restrict__ in = jobs.in[fj] + (live ? rr : 0) + (size_t)g.ndimr * mm;
  double2 *__restrict__ out = jobs.out[fj] + (inr ? rr : 0) + (size_t)g.ndimr * mm;
  const size_t zs = (size_t)g.ndimr * g.ndimth, ks = (size_t)g.ndimr * g.ntchopdim;
  const double inv = 1.0 / (double)f.n;
  fft_any<false>(
      f, tw, s, lgp, [&](int z) { return live ? in[zs * z] : make_double2(0.0, 0.0); },
      [&](int, int k, double2 v) {
        int kk = -1;
        if (k < g.nxchop) kk = k;
        else if (k > f.n - g.nxchop) kk = g.nxchopdim + (k - f.n);
        if (kk >= 0 && inr) out[ks * kk] = make_double2(v.x * inv, v.y * inv);
      });
}

// ---- VERFFT backward: PFF (r, m, k) -> PFP (r, m, z), unscaled; jobs.dz,
// dm: the transform of i k or i m times the input
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_verfft_bwd_any(KGrid g, FftAny f, int lgp, const double2 *__restrict__ tw, TransformJobs jobs, int nj,
                                                        const double *__restrict__ ak) {
  extern __shared__ double2 s[];
  const int P = 1 << lgp, nrb = (g.ndimr + P - 1) >> lgp;
  const int lid = xcd_logical(nrb * g.ntchopdim * nj);
  if (lid < 0) return;
  if (lid == 0 && (int)threadIdx.x < jobs.nzl) jobs.zl[threadIdx.x][0] = 0.0;
  const int bx = lid % nrb, rest = lid / nrb, mm = rest % g.ntchopdim, fj = rest / g.ntchopdim;
  const int rr = (bx << lgp) + (threadIdx.x & (P - 1));
  const bool live = rr < g.nr, inr = rr < g.ndimr;
  const double2 *__restrict__ in = jobs.in[fj] + (live ? rr : 0) + (size_t)g.ndimr * mm;
  double2 *__restrict__ out = jobs.out[fj] + (inr ? rr : 0) + (size_t)g.ndimr * mm;
  const size_t zs = (size_t)g.ndimr * g.ndimth, ks = (size_t)g.ndimr * g.ntchopdim;
  const bool dz = (jobs.dz >> fj) & 1u, dm = (jobs.dm >> fj) & 1u;
  const double mv = (double)(mm * g.minc);
  fft_any<true>(
      f, tw, s, lgp,
      [&](int k) {
        int kk = -1;
        if (k < g.nxchop) kk = k;
        else if (k > f.n - g.nxchop) kk = g.nxchopdim + (k - f.n);
        double2 v = (live && kk >= 0) ? in[ks * kk] : make_double2(0.0, 0.0);
        if (dz) {
          const double kv = kk >= 0 ? ak[mm + (size_t)g.ntchopdim * kk] : 0.0;
          v = make_double2(-kv * v.y, kv * v.x);
        }
        if (dm) v = make_double2(-mv * v.y, mv * v.x);
        return v;
      },
      [&](int, int z, double2 v) {
        if (inr) out[zs * z] = v;
      });
}

// ---- HORFFT forward, in place: PPP slots -> PFP m < NTCHOPDIM (the packed
// real transform's split, as in k_horfft_fwd4).  The results of the last
// stage go back to LDS in place (direct: to the second half), where X_m
// finds Z_m and Z_{NTH-m} through f.pos.
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_horfft_fwd_any(KGrid g, FftAny f, int lgp, const double2 *__restrict__ tw, const double2 *__restrict__ twh, HorJobs jobs) {
  extern __shared__ double2 s[];
  const int P = 1 << lgp, N = f.n, nrb = (g.ndimr + P - 1) >> lgp;
  const int lid = xcd_logical(nrb * g.ndimx * jobs.n);
  if (lid < 0) return;
  const int r0 = (lid % nrb) << lgp, rest = lid / nrb, z = rest % g.ndimx;
  const int p = threadIdx.x & (P - 1), rr = r0 + p;
  const bool live = rr < g.nr;
  double2 *__restrict__ a = jobs.a[rest / g.ndimx] + (size_t)g.ndimr * g.ndimth * z;
  double2 *t = s + (f.direct ? (N << lgp) : 0);
  fft_any<false>(
      f, tw, s, lgp, [&](int j) { return live ? a[rr + (size_t)g.ndimr * j] : make_double2(0.0, 0.0); },
      [&](int pos, int, double2 v) { t[(pos << lgp) + p] = v; });
  __syncthreads();
  const double inv = 1.0 / (double)(2 * N);
  for (int mm = threadIdx.x >> lgp; mm < g.ntchopdim; mm += blockDim.x >> lgp) {
    if (rr >= g.ndimr) break;
    const double2 zm = t[(f.pos[mm] << lgp) + p], zn = t[(f.pos[mm ? N - mm : 0] << lgp) + p];
    const double2 zc = make_double2(zn.x, -zn.y);
    const double2 e = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
    const double2 wd = cmul(twh[mm], csub(zm, zc));  // W^m (Z_m - conj Z_{N-m})
    const double sm = inv * (mm == 0 ? jobs.s0 : jobs.s1);
    double2 x = make_double2((e.x + 0.5 * wd.y) * sm, (e.y - 0.5 * wd.x) * sm);
    if (mm == 0) x.y = 0.0;
    if (mm >= g.ntchop || !live) x = make_double2(0.0, 0.0);
    a[rr + (size_t)g.ndimr * mm] = x;
  }
}

// ---- HORFFT backward, in place: PFP m < NTCHOPDIM -> PPP slots.  The merge
// of k_horfft_bwd4 pairs the slots j and N - j, which both come of X_j and
// X_{N-j}: one thread forms the two in LDS from one load of each.  (Merged on
// the loads of a radix-17 first stage instead, the kernel spilled and took
// 804 us per field at 408x204x608.)
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_horfft_bwd_any(KGrid g, FftAny f, int lgp, const double2 *__restrict__ tw, const double2 *__restrict__ twh, HorJobs jobs) {
  extern __shared__ double2 s[];
  const int P = 1 << lgp, N = f.n, nrb = (g.ndimr + P - 1) >> lgp;
  const int lid = xcd_logical(nrb * g.ndimx * jobs.n);
  if (lid < 0) return;
  const int r0 = (lid % nrb) << lgp, rest = lid / nrb, z = rest % g.ndimx;
  const int p = threadIdx.x & (P - 1), rr = r0 + p;
  const bool live = rr < g.nr, inr = rr < g.ndimr;
  // read and written in place: the loads of a line come before the barrier
  double2 *a = jobs.a[rest / g.ndimx] + (size_t)g.ndimr * g.ndimth * z + (inr ? rr : 0);
  double s0 = jobs.s0, s1 = jobs.s1;
  if (jobs.wr && live) {
    const double w = jobs.wr[rr < g.nr - 1 - rr ? rr : g.nr - 1 - rr];
    s0 *= w;
    s1 *= w;
  }
  const int mmax = g.ntchop < g.ntchopdim ? g.ntchop : g.ntchopdim;
  auto X = [&](int m) {
    const double2 v = (live && m < mmax) ? a[(size_t)g.ndimr * m] : make_double2(0.0, 0.0);
    const double sm = m == 0 ? s0 : s1;
    return make_double2(v.x * sm, m == 0 ? 0.0 : v.y * sm);
  };
  for (int j = threadIdx.x >> lgp; 2 * j <= N; j += blockDim.x >> lgp) {
    // slot j: e + i o, e = X_j + conj X_{N-j}, o = (X_j - conj X_{N-j}) e^{i pi j/N};
    // slot N - j: conj e + i conj o (X_N, Nyquist, is chopped)
    const double2 xm = X(j);
    double2 xc = j > 0 ? X(N - j) : make_double2(0.0, 0.0);
    xc.y = -xc.y;
    const double2 e = cadd(xm, xc), o = rmul<true>(csub(xm, xc), twh[j]);
    s[(j << lgp) + p] = make_double2(e.x - o.y, e.y + o.x);
    if (j > 0 && 2 * j < N) s[((N - j) << lgp) + p] = make_double2(e.x + o.y, o.x - e.y);
  }
  __syncthreads();
  fft_any<true, true>(
      f, tw, s, lgp, [&](int) { return make_double2(0.0, 0.0); },
      [&](int, int j, double2 v) {
        if (inr) a[(size_t)g.ndimr * j] = live ? v : make_double2(0.0, 0.0);
      });
  if (inr && threadIdx.x < P) a[(size_t)g.ndimr * N] = make_double2(0.0, 0.0);
}

// -------------------------------------------------------------------------
// Short lengths (fft_short, N <= 24): each thread sums one result directly from
// the block's staged lines, terms paired by symmetry.  On small grids a launch
// is a chain of latencies, and the kernels above add the look-up of their plan
// to it; on large ones their one butterfly a thread leaves most lanes of a
// block idle.  us, backward and forward together, against the kernels above
// (NR x lines); the line is where the sums' work has eaten the difference:
//                16x4         128x32       200x64       400x256
//   VERFFT 12    4.9   10.1    7.5  12.8    7.7  13.0   10.3  19.8
//          20    6.3    8.8    9.5  11.3    9.6  11.3   15.0  24.5
//          24    6.9    9.0   11.4  11.4   10.5  11.6   17.5  25.9
//   HORFFT 12    5.9    8.9    7.4  10.3    8.2  10.5   17.4  39.3
//          20    7.2   10.0    9.0  11.0   10.2  12.7   26.4  56.1
//          24    7.4   10.1    9.1  11.2   11.1  13.0   33.1  60.1
// s: [position][pencil]; w: the roots.
constexpr int SHORT_MAX = FFT_SHORT, SHORT_P = 32;

// Terms j and N - j of a sum, u w^j + v w^-j: A + i B gathers (u + v) Re w^j and
// (u - v) Im w^j, half the products and the smaller rounding
__device__ __forceinline__ void short_pair(double2 u, double2 v, double2 t, double2 &A, double2 &B) {
  A.x += (u.x + v.x) * t.x;
  A.y += (u.y + v.y) * t.x;
  B.x += (u.x - v.x) * t.y;
  B.y += (u.y - v.y) * t.y;
}

__global__ void __launch_bounds__(256) k_verfft_fwd_short(KGrid g, int N, const double2 *__restrict__ tw, TransformJobs jobs) {
  __shared__ double2 s[SHORT_MAX * SHORT_P], w[SHORT_MAX];
  const int p = threadIdx.x % SHORT_P, i0 = threadIdx.x / SHORT_P, rr = blockIdx.x * SHORT_P + p, mm = blockIdx.y;
  const bool live = rr < g.nr;
  const double2 *__restrict__ in = jobs.in[blockIdx.z] + rr + (size_t)g.ndimr * mm;
  double2 *__restrict__ out = jobs.out[blockIdx.z] + rr + (size_t)g.ndimr * mm;
  if ((int)threadIdx.x < N) w[threadIdx.x] = tw[threadIdx.x];
  for (int z = i0; z < N; z += 256 / SHORT_P)
    s[z * SHORT_P + p] = live ? in[(size_t)g.ndimr * g.ndimth * z] : make_double2(0.0, 0.0);
  __syncthreads();
  if (rr >= g.ndimr) return;
  for (int kk = i0; kk < g.nxchopdim; kk += 256 / SHORT_P) {
    const int k = kk < g.nxchop ? kk : N - (g.nxchopdim - kk);
    double2 A = s[p], B = make_double2(0.0, 0.0);
    int ph = 0;
    for (int z = 1; 2 * z < N; z++) {
      const double2 u = s[z * SHORT_P + p], v = s[(N - z) * SHORT_P + p];
      ph += k;
      if (ph >= N) ph -= N;
      short_pair(u, v, w[ph], A, B);
    }
    if (N % 2 == 0) {
      const double2 u = s[N / 2 * SHORT_P + p];
      A = k % 2 ? csub(A, u) : cadd(A, u);
    }
    out[(size_t)g.ndimr * g.ntchopdim * kk] = make_double2((A.x - B.y) / N, (A.y + B.x) / N);
  }
}

__global__ void __launch_bounds__(256) k_verfft_bwd_short(KGrid g, int N, const double2 *__restrict__ tw, TransformJobs jobs,
                                                          const double *__restrict__ ak) {
  __shared__ double2 s[SHORT_MAX * SHORT_P], w[SHORT_MAX];
  const int p = threadIdx.x % SHORT_P, i0 = threadIdx.x / SHORT_P, rr = blockIdx.x * SHORT_P + p, mm = blockIdx.y;
  const int fj = blockIdx.z, K = g.nxchopdim;
  if (blockIdx.x + blockIdx.y + blockIdx.z == 0 && (int)threadIdx.x < jobs.nzl) jobs.zl[threadIdx.x][0] = 0.0;
  const bool live = rr < g.nr, dz = (jobs.dz >> fj) & 1u, dm = (jobs.dm >> fj) & 1u;
  const double2 *__restrict__ in = jobs.in[fj] + rr + (size_t)g.ndimr * mm;
  double2 *__restrict__ out = jobs.out[fj] + rr + (size_t)g.ndimr * mm;
  if ((int)threadIdx.x < N) w[threadIdx.x] = tw[threadIdx.x];
  for (int kk = i0; kk < K; kk += 256 / SHORT_P) {
    double2 v = live ? in[(size_t)g.ndimr * g.ntchopdim * kk] : make_double2(0.0, 0.0);
    if (dz) {
      const double kv = ak[mm + (size_t)g.ntchopdim * kk];
      v = make_double2(-kv * v.y, kv * v.x);
    }
    if (dm) {
      const double mv = (double)(mm * g.minc);
      v = make_double2(-mv * v.y, mv * v.x);
    }
    s[kk * SHORT_P + p] = v;
  }
  __syncthreads();
  if (rr >= g.ndimr) return;
  for (int z = i0; z < N; z += 256 / SHORT_P) {
    double2 A = s[p], B = make_double2(0.0, 0.0);
    int ph = 0;
    for (int k = 1; k < g.nxchop; k++) {  // k and -k
      ph += z;
      if (ph >= N) ph -= N;
      short_pair(s[k * SHORT_P + p], s[(K - k) * SHORT_P + p], w[ph], A, B);
    }
    out[(size_t)g.ndimr * g.ndimth * z] = make_double2(A.x + B.y, A.y - B.x);
  }
}

// HORFFT: the 2 N real samples of a line (slot j: 2j, 2j + 1) and its modes
// m < NTCHOPDIM, with the roots of order 2 N, in place
__device__ __forceinline__ void short_roots(double2 *w, int N, const double2 *__restrict__ twh) {
  if ((int)threadIdx.x < 2 * N) {
    const int j = threadIdx.x;
    const double2 t = twh[j <= N ? j : j - N];
    w[j] = j <= N ? t : make_double2(-t.x, -t.y);
  }
}
__global__ void __launch_bounds__(256) k_horfft_fwd_short(KGrid g, int N, const double2 *__restrict__ twh, HorJobs jobs) {
  __shared__ double s[2 * SHORT_MAX * SHORT_P];
  __shared__ double2 w[2 * SHORT_MAX];
  const int p = threadIdx.x % SHORT_P, i0 = threadIdx.x / SHORT_P, rr = blockIdx.x * SHORT_P + p;
  const bool live = rr < g.nr;
  double2 *a = jobs.a[blockIdx.z] + rr + (size_t)g.ndimr * g.ndimth * blockIdx.y;
  short_roots(w, N, twh);
  for (int j = i0; j < N; j += 256 / SHORT_P) {
    const double2 v = live ? a[(size_t)g.ndimr * j] : make_double2(0.0, 0.0);
    s[2 * j * SHORT_P + p] = v.x;
    s[(2 * j + 1) * SHORT_P + p] = v.y;
  }
  __syncthreads();
  if (rr >= g.ndimr) return;
  for (int mm = i0; mm < g.ntchopdim; mm += 256 / SHORT_P) {
    double2 x = make_double2(0.0, 0.0);
    if (mm < g.ntchop && live) {
      // samples t, 2 N - t, N - t and N + t together
      const double sg = mm % 2 ? -1.0 : 1.0;
      auto S = [&](int t) { return s[t * SHORT_P + p]; };
      x.x = S(0) + sg * S(N);
      int ph = 0;
      for (int t = 1; 2 * t < N; t++) {
        ph += mm;
        if (ph >= 2 * N) ph -= 2 * N;
        const double a = S(t), b = S(2 * N - t), c = S(N - t), d = S(N + t);
        x = make_double2(x.x + ((a + b) + sg * (c + d)) * w[ph].x, x.y + ((a - b) - sg * (c - d)) * w[ph].y);
      }
      if (N % 2 == 0) {
        const double a = S(N / 2), b = S(N + N / 2);
        ph += mm;
        if (ph >= 2 * N) ph -= 2 * N;
        x = make_double2(x.x + (a + b) * w[ph].x, x.y + (a - b) * w[ph].y);
      }
      const double sm = (mm == 0 ? jobs.s0 : jobs.s1) / (2 * N);
      x = make_double2(x.x * sm, mm == 0 ? 0.0 : x.y * sm);
    }
    a[(size_t)g.ndimr * mm] = x;
  }
}
__global__ void __launch_bounds__(256) k_horfft_bwd_short(KGrid g, int N, const double2 *__restrict__ twh, HorJobs jobs) {
  __shared__ double2 s[SHORT_MAX * SHORT_P], w[2 * SHORT_MAX];
  const int p = threadIdx.x % SHORT_P, i0 = threadIdx.x / SHORT_P, rr = blockIdx.x * SHORT_P + p, M = g.ntchopdim;
  const bool live = rr < g.nr;
  double2 *a = jobs.a[blockIdx.z] + rr + (size_t)g.ndimr * g.ndimth * blockIdx.y;
  const double wr = jobs.wr && live ? jobs.wr[rr < g.nr - 1 - rr ? rr : g.nr - 1 - rr] : 1.0;
  short_roots(w, N, twh);
  for (int mm = i0; mm < M; mm += 256 / SHORT_P) {
    double2 v = make_double2(0.0, 0.0);
    if (live && mm < g.ntchop) {
      const double sm = (mm == 0 ? jobs.s0 : 2.0 * jobs.s1) * wr;  // m >= 1 twice, as m and -m
      v = a[(size_t)g.ndimr * mm];
      v = make_double2(v.x * sm, mm == 0 ? 0.0 : v.y * sm);
    }
    s[mm * SHORT_P + p] = v;
  }
  __syncthreads();
  if (rr >= g.ndimr) return;
  for (int j = i0; j <= N; j += 256 / SHORT_P) {
    double2 x = make_double2(0.0, 0.0);
    if (j < N) {
      int pe = 0, po = 0;  // m 2j and m (2j + 1) mod 2 N
      for (int mm = 0; mm < M; mm++) {
        const double2 c = s[mm * SHORT_P + p];
        x.x += c.x * w[pe].x + c.y * w[pe].y;
        x.y += c.x * w[po].x + c.y * w[po].y;
        pe += 2 * j;
        if (pe >= 2 * N) pe -= 2 * N;
        po += 2 * j + 1;
        if (po >= 2 * N) po -= 2 * N;
      }
    }
    a[(size_t)g.ndimr * j] = x;
  }
}

// Pencils per block (log2): as many of 1..32 as fit 80 KB of LDS (two blocks
// per CU), `copies` buffers of the line; one pencil of 4096 points with a
// second buffer takes 128 KB.  Runs of 8 nodes (128 B) or more up to N = 640.
// (Dynamic LDS up to the device's 160 KB needs no function attribute.)
static int any_lgp(int n, int copies) {
  int lg = 5;
  while (lg > 0 && ((size_t)n << lg) * sizeof(double2) * copies > 80 * 1024) lg--;
  return lg;
}

int fft_any_setup(int n, FftAny *f) {
  FftFactors ff;
  *f = FftAny{};
  f->n = n;
  if (fft_short(n)) return 0;
  if (!fft_factor(n, ff)) return MLG_E_ARG;
  std::vector<int> freq, pos;
  fft_order(ff, freq, pos);
  freq.insert(freq.end(), pos.begin(), pos.end());
  int *d = nullptr;
  MLG_CHECK_HIP(hipMalloc((void **)&d, sizeof(int) * freq.size()));
  f->freq = d;
  f->pos = d + (freq.size() - pos.size());
  MLG_CHECK_HIP(hipMemcpy(d, freq.data(), sizeof(int) * freq.size(), hipMemcpyHostToDevice));
  f->ns = ff.ns;
  f->direct = ff.direct;
  for (int i = 0; i < ff.ns; i++) f->rad[i] = ff.rad[i];
  return 0;
}

int launch_verfft_any(mlg_ctx *c, int n, const TransformJobs &jobs, bool fwd) {
  KGrid g = kgrid(c);
  const FftAny &f = c->fz;
  KScope ks(c, fwd ? K_VERFFT_FWD : K_VERFFT_BWD, n * 16.0 * g.nr * g.ntchopdim * (double)(g.nx + g.nxchopdim));
  if (fft_short(f.n)) {
    const dim3 grid((g.ndimr + SHORT_P - 1) / SHORT_P, g.ntchopdim, n);
    if (fwd) hipLaunchKernelGGL(k_verfft_fwd_short, grid, dim3(256), 0, c->stream, g, f.n, c->d.tw_z, jobs);
    else hipLaunchKernelGGL(k_verfft_bwd_short, grid, dim3(256), 0, c->stream, g, f.n, c->d.tw_z, jobs, c->d.ak);
    MLG_CHECK_HIP(hipGetLastError());
    return 0;
  }
  const int lg = any_lgp(f.n, 1), P = 1 << lg;
  const dim3 grid(xcd_grid((g.ndimr + P - 1) / P * g.ntchopdim * n));
  const size_t lds = sizeof(double2) * ((size_t)f.n << lg);
  if (fwd)
    hipLaunchKernelGGL(k_verfft_fwd_any, grid, dim3(256), lds, c->stream, g, f, lg, c->d.tw_z, jobs, n);
  else
    hipLaunchKernelGGL(k_verfft_bwd_any, grid, dim3(256), lds, c->stream, g, f, lg, c->d.tw_z, jobs, n, c->d.ak);
  MLG_CHECK_HIP(hipGetLastError());
  return 0;
}

int launch_horfft_any(mlg_ctx *c, const HorJobs &jobs, bool fwd) {
  KGrid g = kgrid(c);
  const FftAny &f = c->ft;
  if (fft_short(f.n)) {
    const dim3 grid((g.ndimr + SHORT_P - 1) / SHORT_P, g.ndimx, jobs.n);
    if (fwd) hipLaunchKernelGGL(k_horfft_fwd_short, grid, dim3(256), 0, c->stream, g, f.n, c->d.tw_h, jobs);
    else hipLaunchKernelGGL(k_horfft_bwd_short, grid, dim3(256), 0, c->stream, g, f.n, c->d.tw_h, jobs);
    MLG_CHECK_HIP(hipGetLastError());
    return 0;
  }
  const int copies = fwd && f.direct ? 2 : 1;
  const int lg = any_lgp(f.n, copies), P = 1 << lg;
  const dim3 grid(xcd_grid((g.ndimr + P - 1) / P * g.ndimx * jobs.n));
  const size_t lds = sizeof(double2) * ((size_t)f.n << lg) * copies;
  if (fwd)
    hipLaunchKernelGGL(k_horfft_fwd_any, grid, dim3(256), lds, c->stream, g, f, lg, c->d.tw_t, c->d.tw_h, jobs);
  else
    hipLaunchKernelGGL(k_horfft_bwd_any, grid, dim3(256), lds, c->stream, g, f, lg, c->d.tw_t, c->d.tw_h, jobs);
  MLG_CHECK_HIP(hipGetLastError());
  return 0;
}

}  // namespace mlg
