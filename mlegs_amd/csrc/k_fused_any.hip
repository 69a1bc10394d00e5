// Physical-space products fused with the theta transforms at any planned
// theta length (fused_plan, fft_plan.h): k_fused.hip's products for lengths
// without a register-resident line kernel of their own.
//
// A block owns P adjacent radial lines of one z plane.  Fields come to
// physical space one at a time through LDS (mixed-radix decimation in
// frequency, in place, as k_fft_any.hip); the last stage's butterfly leaves
// R of the line's points in each thread's registers, the same points for
// every field, so the products are formed in registers, and the forward
// transforms run the stages backwards from there.  The next field's loads are
// issued behind the current field's merge; the roots are in LDS, so that no
// stage waits on the memory counter that those loads hold.
//
// In place of ten inverse transforms to memory, the products and four forward
// transforms (k_fft_any.hip): 1.39 ms against 1.94 at NTH = 204, NR = 408, NX =
// 128.  PFP traffic (nine or ten fields in, four out) is 0.16 ms of it; the
// rest is the stages' LDS passes and barriers at two waves a SIMD.
#include "fft_radix.h"
#include "fused_io.h"
#include "mlegs_internal.h"
#include "xcd.h"

namespace mlg {

#pragma clang fp contract(fast)

namespace {

using namespace fftr;

#define MID_RADIX(R_, CALL) \
  switch (R_) {             \
    case 2: CALL(2); break; \
    case 3: CALL(3); break; \
    case 4: CALL(4); break; \
    case 5: CALL(5); break; \
    case 6: CALL(6); break; \
    case 7: CALL(7); break; \
    case 8: CALL(8); break; \
    default: break;         \
  }

struct Lds {
  double2 *tw, *th, *s0, *s1;  // roots W_n^k, e^{-i pi k / n} (k <= n/2), line buffers
};

// middle stage of radix r on blocks of length L, in place in s1: inverse
// (DFT, then roots) or forward (roots, then DFT)
template <int r, bool INV>
__device__ __forceinline__ void mid_stage(int n, int P, int p, int i0, int istep, int L, unsigned magic, const Lds &l) {
  const int M = L / r, step = n / L;
  for (int i = i0; i < n / r; i += istep) {
    const int b = (int)__umulhi((unsigned)i, magic), j = i - b * M;  // i / M
    double2 *x = l.s1 + (b * L + j) * P + p;
    double2 v[r];
#pragma unroll
    for (int q = 0; q < r; q++) v[q] = x[M * q * P];
    if (!INV) {
#pragma unroll
      for (int k = 1; k < r; k++) v[k] = rmul<false>(v[k], l.tw[j * k * step]);
    }
    Dft<r, INV>::run(v, nullptr, 0);
    if (INV) {
#pragma unroll
      for (int k = 1; k < r; k++) v[k] = rmul<true>(v[k], l.tw[j * k * step]);
    }
#pragma unroll
    for (int q = 0; q < r; q++) x[M * q * P] = v[q];
  }
}
template <bool INV>
__device__ __forceinline__ void mid_any(int r, int n, int P, int p, int i0, int istep, int L, unsigned magic, const Lds &l) {
#define C_MID(R_) mid_stage<R_, INV>(n, P, p, i0, istep, L, magic, l)
  MID_RADIX(r, C_MID)
#undef C_MID
}

// the direct stage of length D over the whole line (stride M = n / D):
// inverse s0 -> s1 (sums, then roots), forward s1 -> s0 (roots, then sums);
// outputs k and D - k together
template <bool INV>
__device__ __forceinline__ void direct_stage(int n, int D, int M, int P, int p, int i0, int istep, unsigned magic, const Lds &l) {
  const int H = (D - 1) / 2;
  const double2 *in = INV ? l.s0 : l.s1;
  double2 *out = INV ? l.s1 : l.s0;
  for (int i = i0; i < M * (H + 1); i += istep) {
    const int k = (int)__umulhi((unsigned)i, magic), j = i - k * M;  // i / M
    double2 A = in[j * P + p], B = make_double2(0.0, 0.0);
    int ph = 0;
    for (int q = 1; q <= H; q++) {
      double2 u = in[(j + M * q) * P + p], w = in[(j + M * (D - q)) * P + p];
      if (!INV) {
        u = rmul<false>(u, l.tw[j * q]);
        w = rmul<false>(w, l.tw[j * (D - q)]);
      }
      ph += k;
      if (ph >= D) ph -= D;
      const double2 t = l.tw[ph * M];
      A.x += (u.x + w.x) * t.x;
      A.y += (u.y + w.y) * t.x;
      B.x += (u.x - w.x) * t.y;
      B.y += (u.y - w.y) * t.y;
    }
    const double2 jb = INV ? make_double2(B.y, -B.x) : make_double2(-B.y, B.x);
    double2 y = cadd(A, jb), yc = csub(A, jb);
    if (INV) {
      y = rmul<true>(y, l.tw[j * k]);
      if (k > 0) yc = rmul<true>(yc, l.tw[j * (D - k)]);
    }
    out[(j + M * k) * P + p] = y;
    if (k > 0) out[(j + M * (D - k)) * P + p] = yc;
  }
}

}  // namespace

template <int R, bool LINEAR>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
k_fused_any(KGrid g, FusedAny f, const double *__restrict__ rsq, const double2 *__restrict__ tw,
            const double2 *__restrict__ twh, FusedIO io, double two_omega, double n2) {
  if (blockIdx.x == 0 && threadIdx.x == 0 && io.zl) io.zl[0] = 0.0;
  extern __shared__ double2 sm[];
  constexpr int NP = R / 2 + 1;        // pairs of a line a thread merges
  const int n = f.n, P = f.P, nb = n / R;
  const int nrb = (g.ndimr + P - 1) / P;
  const int lid = xcd_logical(nrb * g.ndimx);
  if (lid < 0) return;
  const int z = lid / nrb, r0 = (lid - z * nrb) * P, tid = threadIdx.x;
  Lds l;
  l.tw = sm;
  l.th = sm + n;
  l.s1 = l.th + n / 2 + 1;
  l.s0 = f.D > 1 ? l.s1 + n * P : l.s1;
  for (int i = tid; i < n; i += blockDim.x) l.tw[i] = tw[i];
  for (int i = tid; i <= n / 2; i += blockDim.x) l.th[i] = twh[i];
  // lanes over the lines of the block, then its points; the threads past the
  // last whole set of lines idle
  const int istep = blockDim.x / P, p = tid % P, b = tid / P, i0 = b < istep ? b : n;
  const bool own = b < nb && b < istep;
  const int rr = r0 + p;
  const bool live = rr < g.nr && b < istep, inr = rr < g.ndimr;
  const int mmax = g.ntchop < g.ntchopdim ? g.ntchop : g.ntchopdim;
  const size_t off = (size_t)g.ndimr * g.ndimth * z + (inr ? rr : 0);
  const double r2 = live ? rsq[rr] : 1.0;

  double2 xa[NP], xb[NP];
  auto fetch = [&](int q) {
    const double2 *src = io.in[q] + off;
#pragma unroll
    for (int u = 0; u < NP; u++) {
      const int j = i0 + u * istep;
      xa[u] = xb[u] = make_double2(0.0, 0.0);
      if (live && 2 * j <= n && j < mmax) xa[u] = src[(size_t)g.ndimr * j];
      if (live && j > 0 && 2 * j <= n && n - j < mmax) xb[u] = src[(size_t)g.ndimr * (n - j)];
    }
  };
  // slots j and n - j from X_j and X_{n-j} (k_horfft_bwd_any's merge)
  auto merge = [&]() {
#pragma unroll
    for (int u = 0; u < NP; u++) {
      const int j = i0 + u * istep;
      if (2 * j > n) continue;
      double2 xm = xa[u];
      if (j == 0) xm.y = 0.0;
      const double2 xc = make_double2(xb[u].x, -xb[u].y);
      const double2 e = cadd(xm, xc), o = rmul<true>(csub(xm, xc), l.th[j]);
      l.s0[j * P + p] = make_double2(e.x - o.y, e.y + o.x);
      if (j > 0 && 2 * j < n) l.s0[(n - j) * P + p] = make_double2(e.x + o.y, o.x - e.y);
    }
  };
  // the field fetched before to the thread's points v; next: the field fetched behind it
  auto inverse = [&](int next, double2(&v)[R]) {
    __syncthreads();  // the buffers' last readers are done (first: the roots are there)
    merge();
    if (next >= 0) fetch(next);
    __syncthreads();
    int L = n;
    if (f.D > 1) {
      direct_stage<true>(n, f.D, f.md, P, p, i0, istep, f.magic_d, l);
      __syncthreads();
      L = f.md;
    }
    for (int s = 0; s < f.nmid; s++) {
      mid_any<true>(f.mid[s], n, P, p, i0, istep, L, f.magic[s], l);
      __syncthreads();
      L /= f.mid[s];
    }
    if (own) {
#pragma unroll
      for (int k = 0; k < R; k++) v[k] = l.s1[(b * R + k) * P + p];
    } else {
#pragma unroll
      for (int k = 0; k < R; k++) v[k] = make_double2(0.0, 0.0);
    }
    Dft<R, true>::run(v, nullptr, 0);
  };
  auto forward = [&](double2(&v)[R], int q) {
    Dft<R, false>::run(v, nullptr, 0);
    __syncthreads();
    if (own) {
#pragma unroll
      for (int k = 0; k < R; k++) l.s1[(b * R + k) * P + p] = v[k];
    }
    __syncthreads();
    int L = R;
    for (int s = f.nmid - 1; s >= 0; s--) {
      L *= f.mid[s];
      mid_any<false>(f.mid[s], n, P, p, i0, istep, L, f.magic[s], l);
      __syncthreads();
    }
    if (f.D > 1) {
      direct_stage<false>(n, f.D, f.md, P, p, i0, istep, f.magic_d, l);
      __syncthreads();
    }
    double2 *dst = io.out[q] + off;
    const double inv = 1.0 / (double)(2 * n);
    for (int mm = i0; mm < g.ntchopdim; mm += istep) {
      if (!inr) break;
      const double2 zm = l.s0[mm * P + p], zn = l.s0[(mm ? n - mm : 0) * P + p];
      const double2 zc = make_double2(zn.x, -zn.y);
      // e^{-i pi m / n}; beyond n / 2 it is -conj of that at n - m
      const double2 t0 = l.th[2 * mm <= n ? mm : n - mm];
      const double2 t = make_double2(2 * mm <= n ? t0.x : -t0.x, t0.y);
      const double2 wd = cmul(t, csub(zm, zc));
      double2 x = make_double2((0.5 * (zm.x + zc.x) + 0.5 * wd.y) * inv, (0.5 * (zm.y + zc.y) - 0.5 * wd.x) * inv);
      if (mm == 0) x.y = 0.0;
      if (mm >= g.ntchop || rr >= g.nr) x = make_double2(0.0, 0.0);
      dst[(size_t)g.ndimr * mm] = x;
    }
  };

  // k_fused_products_256's field order: ror, rop, oz are read before the
  // results that overwrite them are written
  double2 A[R], B[R], C[R], U[R], V[R], T[R], Y[R];
  fetch(0);
  inverse(1, A);  // rur
  inverse(2, B);  // rup
  inverse(5, C);  // uz
  inverse(3, T);  // oz
#pragma unroll
  for (int i = 0; i < R; i++) {
    U[i] = make_double2(B[i].x * T[i].x, B[i].y * T[i].y);
    V[i] = make_double2(A[i].x * T[i].x, A[i].y * T[i].y);
  }
  inverse(4, T);  // ror: Y = uz ror - rur oz, V = rup ror
#pragma unroll
  for (int i = 0; i < R; i++) {
    Y[i] = make_double2(C[i].x * T[i].x - V[i].x, C[i].y * T[i].y - V[i].y);
    V[i] = make_double2(B[i].x * T[i].x, B[i].y * T[i].y);
  }
  inverse(LINEAR ? 9 : 6, T);  // rop: X = rup oz - uz rop, Z = (rur rop - rup ror) / r^2
#pragma unroll
  for (int i = 0; i < R; i++) {
    U[i] = make_double2(U[i].x - C[i].x * T[i].x, U[i].y - C[i].y * T[i].y);
    V[i] = make_double2((A[i].x * T[i].x - V[i].x) / r2, (A[i].y * T[i].y - V[i].y) / r2);
    if (LINEAR) U[i] = make_double2(U[i].x + two_omega * B[i].x, U[i].y + two_omega * B[i].y);
  }
  forward(U, 0);
#pragma unroll
  for (int i = 0; i < R; i++) {
    T[i] = Y[i];
    if (LINEAR) T[i] = make_double2(T[i].x - two_omega * A[i].x, T[i].y - two_omega * A[i].y);
  }
  forward(T, 1);
  if (LINEAR) {
    inverse(6, T);  // W: N_z = Z - W
#pragma unroll
    for (int i = 0; i < R; i++) V[i] = make_double2(V[i].x - T[i].x, V[i].y - T[i].y);
  }
  forward(V, 2);
  inverse(7, T);  // rbr
#pragma unroll
  for (int i = 0; i < R; i++) A[i] = make_double2(A[i].x * T[i].x, A[i].y * T[i].y);
  inverse(8, T);  // rbp
#pragma unroll
  for (int i = 0; i < R; i++) A[i] = make_double2(A[i].x + B[i].x * T[i].x, A[i].y + B[i].y * T[i].y);
  inverse(-1, T);  // bz: N_b = -(T / r^2 + uz bz) (+ Nbar^2 uz)
#pragma unroll
  for (int i = 0; i < R; i++) {
    const double vr = A[i].x / r2 + C[i].x * T[i].x, vi = A[i].y / r2 + C[i].y * T[i].y;
    A[i] = make_double2(-vr, -vi);
    if (LINEAR) A[i] = make_double2(A[i].x + n2 * C[i].x, A[i].y + n2 * C[i].y);
  }
  forward(A, 3);
}

int fused_any_setup(int nth, FusedAny *f) {
  FusedPlan q;
  *f = FusedAny{};
  if (!fused_plan(nth, q)) return 0;
  f->n = q.n, f->R = q.R, f->D = q.D, f->nmid = q.nmid, f->P = q.P, f->T = q.T;
  // i / M = umulhi(i, ceil(2^32 / M)) exactly for i, M < 2^16; M >= 2 in every stage before the last
  auto magic = [](int m) { return (unsigned)(((1ull << 32) + m - 1) / m); };
  int L = q.n / q.D;
  f->md = L;
  f->magic_d = magic(L);
  for (int i = 0; i < q.nmid; i++) {
    f->mid[i] = q.mid[i];
    L /= q.mid[i];
    f->magic[i] = magic(L);
  }
  f->lds = fused_lds(q) * (long)sizeof(double2);
  return 0;
}

int launch_fused_any(mlg_ctx *c, const FusedIO &io, double two_omega, double n2, int linear) {
  KGrid g = kgrid(c);
  const FusedAny &f = c->fp;
  const dim3 grid(xcd_grid((g.ndimr + f.P - 1) / f.P * g.ndimx));
#define L_ANY(R_)                                                                                                      \
  case R_:                                                                                                             \
    if (linear)                                                                                                        \
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fused_any<R_, true>), grid, dim3(f.T), f.lds, c->stream, g, f, c->d.r,      \
                         c->d.tw_t, c->d.tw_h, io, two_omega, n2);                                                     \
    else                                                                                                               \
      hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fused_any<R_, false>), grid, dim3(f.T), f.lds, c->stream, g, f, c->d.r,     \
                         c->d.tw_t, c->d.tw_h, io, two_omega, n2);                                                     \
    break
  switch (f.R) {
    L_ANY(2);
    L_ANY(3);
    L_ANY(4);
    L_ANY(5);
    L_ANY(6);
    default: return MLG_E_ARG;
  }
#undef L_ANY
  MLG_CHECK_HIP(hipGetLastError());
  return 0;
}

}  // namespace mlg
