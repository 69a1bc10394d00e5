// Nonlinear terms in physical space without physical-space fields in HBM.
//
// CALC_BOUSSI_FORCE / CALC_BOUSSI_NONLIN (src/mod_boussinesq.f90:235-410)
// take nine fields to physical space (HORFFT backward), form u x omega and
// u . grad b there (VPRODSUB/VDOTPSUB, src/mod_legops.f90:1972-2232, plus
// FORCE's linear terms) and bring four results back (HORFFT forward).  The
// kernels here do all of that for some radial pencils of one z plane at a
// time, reading the inputs in PFP (r, m, z) and writing the outputs in PFP:
// the physical theta lines live only in registers and LDS.
//   products: X = rup oz - uz rop (+ 2 Omega rup), Y = uz ror - rur oz
//     (- 2 Omega rur), Z = (rur rop - rup ror) / r^2 (- W), N_b = -((rur rbr +
//     rup rbp) / r^2 + uz bz) (+ Nbar^2 uz)
//   powers of two up to 512: lines in the registers of 1 .. 64 lanes, all
//     fields of a line in one wave (k_fused_products_256, k_fused_products_reg)
//     or one wave a field (k_fused_products_wide); launch_line has the rule
//   every other length: k_fused_any.hip
// The products are the separate kernels' operations, in the same order; the
// transforms may factor their length in another way than the separate HORFFT.
#include "fused_io.h"
#include "mlegs_internal.h"
#include "xcd.h"

namespace mlg {

// The theta transforms round like any FFT (not operation for operation like
// a reference library): products and sums may contract to FMAs here.
#pragma clang fp contract(fast)

__device__ __forceinline__ double2 fz_cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ double2 fz_conj(double2 a) { return make_double2(a.x, -a.y); }

// ---------------------------------------------------------------------------
// NTH = 256: register-resident variant.
//
// 32 lanes own one theta line (two lines per wave, eight adjacent radial
// nodes per block).  Each lane keeps 8 of the line's 256 physical points in
// registers, at the same positions for every field, so the products are
// formed in registers and only the transposes of the transforms use LDS.
// The 256-point transform is 8 x 8 x 4:
//   j = 32 a + b (lane b holds a = 0..7)      -> 8-point DFT over a, twiddle
//   exchange to lane 4 c + f (holds e = 0..7)  -> 8-point DFT over e, twiddle
//   exchange to lane 4 c + gh (holds f = 0..3 for g = gh, gh + 4)
//                                               -> 4-point DFTs over f
// so lane 4 c + gh ends with the points k = c + 8 g + 64 h, h = 0..3.  The
// forward transform runs the same stages backwards with conjugate roots.
// Waves never wait for one another; the LDS of a line is touched only by
// its own 32 lanes.
// ---------------------------------------------------------------------------
namespace w256 {

constexpr int N = 256;
constexpr int LP = 288;  // LDS double2 per line (two exchange layouts, padded against bank conflicts)
__device__ __forceinline__ int e1(int c, int b) { return c * 36 + b; }
__device__ __forceinline__ int e2(int c, int f, int g) { return c * 36 + f * 9 + g; }

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Per-lane twiddles, copied to LDS once per block:
//   t1[32 c + b] = W_N^{b c}, t2[4 g + f] = W_N^{8 f g}, th[k] = exp(-i pi k / N)
struct Ctx {
  const double2 *t1, *t2, *th;
  double2 *s;                       // LDS of this line
  int b;                            // lane within the line
};

// 8- and 4-point DFTs with the roots exp(S 2 pi i k / R) written out:
// multiplications by 1 and +-i are exact moves, exp(+-i pi/4) uses sqrt(1/2).
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
template <int S>
__device__ __forceinline__ double2 mul_si(double2 d) {  // (S i) d
  return S > 0 ? make_double2(-d.y, d.x) : make_double2(d.y, -d.x);
}
template <int S>
__device__ __forceinline__ void dft4s(double2 (&y)[4]) {
  const double2 a = cadd(y[0], y[2]), b = csub(y[0], y[2]), c = cadd(y[1], y[3]), d = mul_si<S>(csub(y[1], y[3]));
  y[0] = cadd(a, c);
  y[1] = cadd(b, d);
  y[2] = csub(a, c);
  y[3] = csub(b, d);
}
template <int S>
__device__ __forceinline__ void dft8s(double2 (&x)[8]) {
  constexpr double h = 0.70710678118654752440;  // sqrt(1/2)
  double2 e[4] = {x[0], x[2], x[4], x[6]}, o[4] = {x[1], x[3], x[5], x[7]};
  dft4s<S>(e);
  dft4s<S>(o);
  double2 t[4];
  t[0] = o[0];
  t[1] = S > 0 ? make_double2(h * (o[1].x - o[1].y), h * (o[1].y + o[1].x))
               : make_double2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));
  t[2] = mul_si<S>(o[2]);
  t[3] = S > 0 ? make_double2(h * (-o[3].x - o[3].y), h * (o[3].x - o[3].y))
               : make_double2(h * (o[3].y - o[3].x), h * (-o[3].y - o[3].x));
#pragma unroll
  for (int k = 0; k < 4; k++) {
    x[k] = cadd(e[k], t[k]);
    x[k + 4] = csub(e[k], t[k]);
  }
}

// dft8s for inputs with x[3] = x[4] = 0 (the unused slots of a spectrum
// with fewer than 96 modes): the additions of those zeros are left out.
template <int S>
__device__ __forceinline__ void dft8s_z34(double2 (&x)[8]) {
  constexpr double h = 0.70710678118654752440;
  // even part {x0, x2, 0, x6}, odd part {x1, 0, x5, x7}
  double2 e[4], o[4];
  {
    const double2 c = cadd(x[2], x[6]), d = mul_si<S>(csub(x[2], x[6]));
    e[0] = cadd(x[0], c);
    e[1] = cadd(x[0], d);
    e[2] = csub(x[0], c);
    e[3] = csub(x[0], d);
  }
  {
    const double2 a = cadd(x[1], x[5]), b = csub(x[1], x[5]), d = mul_si<-S>(x[7]);
    o[0] = cadd(a, x[7]);
    o[1] = cadd(b, d);
    o[2] = csub(a, x[7]);
    o[3] = csub(b, d);
  }
  double2 t[4];
  t[0] = o[0];
  t[1] = S > 0 ? make_double2(h * (o[1].x - o[1].y), h * (o[1].y + o[1].x))
               : make_double2(h * (o[1].x + o[1].y), h * (o[1].y - o[1].x));
  t[2] = mul_si<S>(o[2]);
  t[3] = S > 0 ? make_double2(h * (-o[3].x - o[3].y), h * (o[3].x - o[3].y))
               : make_double2(h * (o[3].y - o[3].x), h * (-o[3].y - o[3].x));
#pragma unroll
  for (int k = 0; k < 4; k++) {
    x[k] = cadd(e[k], t[k]);
    x[k + 4] = csub(e[k], t[k]);
  }
}

__device__ __forceinline__ double2 cj(double2 w, bool inv) {
  if (inv) w.y = -w.y;
  return w;
}

// Both terms of the Hermitian merge (truncations past 3/8 of NTH): xm = X[j],
// xc = conj X[N-j], th = exp(-i pi j / N)
__device__ __forceinline__ double2 merge_full(double2 xm, double2 xc, double2 th) {
  const double2 e = cadd(xm, xc), o = fz_cmul(csub(xm, xc), fz_conj(th));
  return make_double2(e.x - o.y, e.y + o.x);
}

// HORFFT backward of one PFP line (element m at src[lo + ndimr m], src the
// same for the whole block); lane b ends with the physical points
// P[c + 8 (gh + 4 s) + 64 h] in v[4 s + h], c = b >> 2, gh = b & 3.
// Without FULL, NTCHOPDIM <= MMAX96: only a = 0..2 hold modes, a = 5..7
// partners.
constexpr int MMAX96 = 96;
template <bool FULL>
__device__ __forceinline__ void inverse(const Ctx &x, const KGrid &g, const double2 *__restrict__ src, int lo,
                                        bool live, double2 (&v)[8]) {
  const int b = x.b, mmax = g.ntchopdim;
  // branch-free: masked lanes load row 0 and discard it
  auto X = [&](int m, bool use) -> double2 {
    use = use && live && m < g.ntchop;
    double2 t = src[lo + (use ? g.ndimr * m : 0)];
    if (!use) t = make_double2(0.0, 0.0);
    if (m == 0) t.y = 0.0;
    return t;
  };
  // Hermitian merge: with e = X[j] + conj X[N-j], d = X[j] - conj X[N-j],
  // the point is e + i d conj(th[j]), th[j] = exp(-i pi j / N).  Only one of
  // the two terms is present: X[j] (j < 96) times 1 + i conj(th[j]), or
  // conj X[N-j] (j >= 160) times 1 - i conj(th[j]) = 1 + i th[N-j].
#pragma unroll
  for (int a = 0; a < 8; a++) {
    if (!FULL && (a == 3 || a == 4)) {
      v[a] = make_double2(0.0, 0.0);
      continue;
    }
    const int j = 32 * a + b, jc = N - j;
    if constexpr (FULL) {
      v[a] = merge_full(X(j, j < mmax), fz_conj(X(jc, j > 0 && jc < mmax)), x.th[j]);
      continue;
    }
    const double2 t = x.th[a < 3 ? j : jc];
    const double2 xv = a < 3 ? X(j, j < mmax) : fz_conj(X(jc, jc < mmax));
    const double2 q = a < 3 ? make_double2(1.0 + t.y, t.x) : make_double2(1.0 - t.y, t.x);
    v[a] = fz_cmul(xv, q);
  }
  if constexpr (FULL) dft8s<1>(v);
  else dft8s_z34<1>(v);
  // twiddles W^0 = 1 multiply exactly
#pragma unroll
  for (int c = 1; c < 8; c++) v[c] = fz_cmul(v[c], cj(x.t1[32 * c + b], true));
  // exchange 1: lane b holds y_b[c]; lane 4 c + f takes y_{4 e + f}[c]
#pragma unroll
  for (int c = 0; c < 8; c++) x.s[e1(c, b)] = v[c];
  wave_sync();
  const int c0 = b >> 2, f0 = b & 3;
#pragma unroll
  for (int e = 0; e < 8; e++) v[e] = x.s[e1(c0, 4 * e + f0)];
  wave_sync();
  dft8s<1>(v);
#pragma unroll
  for (int gg = 1; gg < 8; gg++) v[gg] = fz_cmul(v[gg], cj(x.t2[4 * gg + f0], true));
  // exchange 2: lane 4 c + f holds z_{c,f}[g]; lane 4 c + gh takes f = 0..3 of g = gh, gh + 4
#pragma unroll
  for (int gg = 0; gg < 8; gg++) x.s[e2(c0, f0, gg)] = v[gg];
  wave_sync();
  double2 t[2][4];
#pragma unroll
  for (int sg = 0; sg < 2; sg++)
#pragma unroll
    for (int f = 0; f < 4; f++) t[sg][f] = x.s[e2(c0, f, f0 + 4 * sg)];
  wave_sync();
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
    dft4s<1>(t[sg]);
#pragma unroll
    for (int h = 0; h < 4; h++) v[4 * sg + h] = t[sg][h];
  }
}

// HORFFT forward of this lane's physical points v (positions as left by
// `inverse`) into one PFP line (element m at dst[lo + ndimr m]).
template <bool FULL>
__device__ __forceinline__ void forward(const Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *__restrict__ dst,
                                        int lo, bool inr, bool live) {
  const int b = x.b, c0 = b >> 2, f0 = b & 3;
  double2 t[2][4];
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
#pragma unroll
    for (int h = 0; h < 4; h++) t[sg][h] = v[4 * sg + h];
    dft4s<-1>(t[sg]);
    const int gg = f0 + 4 * sg;
#pragma unroll
    for (int f = 1; f < 4; f++) t[sg][f] = fz_cmul(t[sg][f], x.t2[4 * gg + f]);
  }
#pragma unroll
  for (int sg = 0; sg < 2; sg++)
#pragma unroll
    for (int f = 0; f < 4; f++) x.s[e2(c0, f, f0 + 4 * sg)] = t[sg][f];
  wave_sync();
  double2 u[8];
#pragma unroll
  for (int gg = 0; gg < 8; gg++) u[gg] = x.s[e2(c0, f0, gg)];
  wave_sync();
  dft8s<-1>(u);
#pragma unroll
  for (int e = 0; e < 8; e++) x.s[e1(c0, 4 * e + f0)] = u[e];
  wave_sync();
#pragma unroll
  for (int c = 0; c < 8; c++) u[c] = x.s[e1(c, b)];
  wave_sync();
#pragma unroll
  for (int c = 1; c < 8; c++) u[c] = fz_cmul(u[c], x.t1[32 * c + b]);
  dft8s<-1>(u);
  // u[a] = Y[32 a + b]; the Hermitian split pairs Y[m] with Y[N - m],
  // which lane (32 - b) mod 32 holds at a' = 7 - a (lane 0: a' = (8 - a) mod 8)
  const double den = (double)(2 * N);
  const int src = (32 - b) & 31;
#pragma unroll
  for (int a = 0; a < (FULL ? 8 : 3); a++) {
    if (32 * a >= g.ntchopdim) break;
    const int m = 32 * a + b;
    double2 pc;
    pc.x = __shfl(u[7 - a].x, src, 32);
    pc.y = __shfl(u[7 - a].y, src, 32);
    if (b == 0) pc = u[(8 - a) & 7];
    if (m < g.ntchopdim && inr) {
      double2 zm = u[a], zc = fz_conj(pc);
      double2 e = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
      double2 d = make_double2(zm.x - zc.x, zm.y - zc.y);
      double2 wd = fz_cmul(x.th[m], d);
      double2 o = make_double2(e.x + 0.5 * wd.y, e.y - 0.5 * wd.x);
      o = make_double2(o.x / den, o.y / den);
      if (m == 0) o.y = 0.0;
      if (m >= g.ntchop || !live) o = make_double2(0.0, 0.0);
      dst[lo + g.ndimr * m] = o;
    }
  }
}

}  // namespace w256

// The products are the separate kernels' floating-point operations.
// The outputs r N_r, r N_theta, N_z overwrite ror, rop, oz in the callers,
// so all three are read before the first of them is written.  The fields go
// to physical space one at a time; at most five stay in registers, and one
// finished product (Y) waits in LDS.
template <bool LINEAR>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_fused_products_256(KGrid g, const double *__restrict__ rsq, const double2 *tw, const double2 *twh, FusedIO io,
                     double two_omega, double n2) {
  if (blockIdx.x == 0 && threadIdx.x == 0 && io.zl) io.zl[0] = 0.0;
  using namespace w256;
  __shared__ double2 S[8 * LP];
  __shared__ double2 Y[8 * N];  // [line][point i][lane]
  __shared__ double2 T1[256], T2[32], TH[N + 1];
  const int nrb = (g.ndimr + 7) / 8;
  const int lid = xcd_logical(nrb * g.ndimx);
  if (lid < 0) return;
  {
    const int q = threadIdx.x;
    T1[q] = tw[(q & 31) * (q >> 5)];
    if (q < 32) T2[q] = tw[8 * (q & 3) * (q >> 2)];
    TH[q] = twh[q];
    if (q == 0) TH[N] = twh[N];
  }
  __syncthreads();
  const int z = lid / nrb, line = threadIdx.x >> 5;
  const int rr = (lid % nrb) * 8 + line;
  const bool inr = rr < g.ndimr, live = rr < g.nr;
  Ctx x;
  x.t1 = T1;
  x.t2 = T2;
  x.th = TH;
  x.s = S + line * LP;
  x.b = threadIdx.x & 31;
  double2 *ys = Y + line * N + x.b;
  const size_t off = (size_t)(rr - line) + (size_t)g.ndimr * g.ndimth * z;  // same for the block
  const int lo = inr ? line : 0;
  auto in = [&](int q) { return io.in[q] + off; };
  auto out = [&](int q) { return io.out[q] + off; };
  const double r2 = live ? rsq[rr] : 1.0;

  double2 A[8], B[8], C[8], U[8], V[8], T[8];
  inverse<false>(x, g, in(0), lo, live, A);  // rur
  inverse<false>(x, g, in(1), lo, live, B);  // rup
  inverse<false>(x, g, in(2), lo, live, C);  // uz
  // oz: U = rup oz, V = rur oz
  inverse<false>(x, g, in(5), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    U[i] = make_double2(B[i].x * T[i].x, B[i].y * T[i].y);
    V[i] = make_double2(A[i].x * T[i].x, A[i].y * T[i].y);
  }
  // ror: Y = uz ror - rur oz (to LDS); V = rup ror
  inverse<false>(x, g, in(3), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    ys[32 * i] = make_double2(C[i].x * T[i].x - V[i].x, C[i].y * T[i].y - V[i].y);
    V[i] = make_double2(B[i].x * T[i].x, B[i].y * T[i].y);
  }
  // rop: X = rup oz - uz rop in U; Z = (rur rop - rup ror) / r^2 in V
  inverse<false>(x, g, in(4), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    U[i] = make_double2(U[i].x - C[i].x * T[i].x, U[i].y - C[i].y * T[i].y);
    V[i] = make_double2((A[i].x * T[i].x - V[i].x) / r2, (A[i].y * T[i].y - V[i].y) / r2);
  }
  // ror, rop, oz are read: the outputs may now overwrite them
  if (LINEAR) {
#pragma unroll
    for (int i = 0; i < 8; i++) U[i] = make_double2(U[i].x + two_omega * B[i].x, U[i].y + two_omega * B[i].y);
  }
  forward<false>(x, g, U, out(0), lo, inr, live);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    T[i] = ys[32 * i];
    if (LINEAR) T[i] = make_double2(T[i].x - two_omega * A[i].x, T[i].y - two_omega * A[i].y);
  }
  forward<false>(x, g, T, out(1), lo, inr, live);
  if (LINEAR) {
    // W: N_z = Z - W
    inverse<false>(x, g, in(9), lo, live, T);
#pragma unroll
    for (int i = 0; i < 8; i++) V[i] = make_double2(V[i].x - T[i].x, V[i].y - T[i].y);
  }
  forward<false>(x, g, V, out(2), lo, inr, live);
  // rbr, rbp: A = rur rbr + rup rbp
  inverse<false>(x, g, in(6), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) A[i] = make_double2(A[i].x * T[i].x, A[i].y * T[i].y);
  inverse<false>(x, g, in(7), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) A[i] = make_double2(A[i].x + B[i].x * T[i].x, A[i].y + B[i].y * T[i].y);
  // bz: N_b = -(T / r^2 + uz bz) (+ Nbar^2 uz)
  inverse<false>(x, g, in(8), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const double vr = A[i].x / r2 + C[i].x * T[i].x, vi = A[i].y / r2 + C[i].y * T[i].y;
    double2 nb = make_double2(-vr, -vi);
    if (LINEAR) nb = make_double2(nb.x + n2 * C[i].x, nb.y + n2 * C[i].y);
    A[i] = nb;
  }
  forward<false>(x, g, A, out(3), lo, inr, live);
}

// ---------------------------------------------------------------------------
// NTH = 128: register-resident variant.
//
// 16 lanes own one theta line (four lines per wave, sixteen adjacent radial
// nodes per block).  Each lane keeps 8 of the line's 128 points of every
// field in registers.  The 128-point transform is 8 x 4 x 4:
//   j = 16 a + b (lane b holds a = 0..7)         -> 8-point DFT over a, twiddle
//   exchange: lane 4 c2 + f (b = 4 e + f) holds e = 0..3 of c = c2, c2 + 4
//                                                 -> 4-point DFTs over e, twiddle
//   exchange: lane 4 c2 + g holds f = 0..3 of c = c2, c2 + 4
//                                                 -> 4-point DFTs over f
// so lane 4 c2 + g ends with the points k = c + 8 g + 32 h, c = c2, c2 + 4,
// h = 0..3.  The forward transform runs the stages backwards with
// conjugate roots.  Same products, waves and LDS discipline as NTH = 256.
// ---------------------------------------------------------------------------
namespace w128 {

constexpr int N = 128;
constexpr int LP = 160;  // LDS double2 per line (the two exchange layouts, padded against bank conflicts)
constexpr int MMAX48 = 48;  // NTCHOPDIM bound: slots a = 3, 4 hold no mode
__device__ __forceinline__ int e1(int c, int b) { return c * 20 + b; }
__device__ __forceinline__ int e2(int c, int f, int g) { return c * 20 + f * 5 + g; }
using w256::cadd;
using w256::cj;
using w256::csub;
using w256::dft4s;
using w256::dft8s;
using w256::merge_full;
using w256::dft8s_z34;
using w256::wave_sync;
using w256::Ctx;  // t1[16 c + b] = W_N^{b c}, t2[4 g + f] = W_N^{8 f g}, th[k] = exp(-i pi k / N)

// HORFFT backward of one PFP line (element m at src[lo + ndimr m]); lane b
// ends with the physical points P[c + 8 g + 32 h] in v[4 s + h], c = c2 + 4 s,
// c2 = b >> 2, g = b & 3.
template <bool FULL>
__device__ __forceinline__ void inverse(const Ctx &x, const KGrid &g, const double2 *__restrict__ src, int lo,
                                        bool live, double2 (&v)[8]) {
  const int b = x.b, mmax = g.ntchopdim;
  auto X = [&](int m, bool use) -> double2 {
    use = use && live && m < g.ntchop;
    double2 t = src[lo + (use ? g.ndimr * m : 0)];
    if (!use) t = make_double2(0.0, 0.0);
    if (m == 0) t.y = 0.0;
    return t;
  };
  // Hermitian merge with one term per point, as at NTH = 256
#pragma unroll
  for (int a = 0; a < 8; a++) {
    if (!FULL && (a == 3 || a == 4)) {
      v[a] = make_double2(0.0, 0.0);
      continue;
    }
    const int j = 16 * a + b, jc = N - j;
    if constexpr (FULL) {
      v[a] = merge_full(X(j, j < mmax), fz_conj(X(jc, j > 0 && jc < mmax)), x.th[j]);
      continue;
    }
    const double2 t = x.th[a < 3 ? j : jc];
    const double2 xv = a < 3 ? X(j, j < mmax) : fz_conj(X(jc, jc < mmax));
    const double2 q = a < 3 ? make_double2(1.0 + t.y, t.x) : make_double2(1.0 - t.y, t.x);
    v[a] = fz_cmul(xv, q);
  }
  if constexpr (FULL) dft8s<1>(v);
  else dft8s_z34<1>(v);
#pragma unroll
  for (int c = 1; c < 8; c++) v[c] = fz_cmul(v[c], cj(x.t1[16 * c + b], true));
  // exchange 1: lane b holds y_b[c]; lane 4 c2 + f takes y_{4 e + f}[c], c = c2, c2 + 4
#pragma unroll
  for (int c = 0; c < 8; c++) x.s[e1(c, b)] = v[c];
  wave_sync();
  const int c2 = b >> 2, f0 = b & 3;
  double2 t[2][4];
#pragma unroll
  for (int sg = 0; sg < 2; sg++)
#pragma unroll
    for (int e = 0; e < 4; e++) t[sg][e] = x.s[e1(c2 + 4 * sg, 4 * e + f0)];
  wave_sync();
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
    dft4s<1>(t[sg]);
#pragma unroll
    for (int gg = 1; gg < 4; gg++) t[sg][gg] = fz_cmul(t[sg][gg], cj(x.t2[4 * gg + f0], true));
  }
  // exchange 2: lane 4 c2 + f holds z_{c,f}[g]; lane 4 c2 + g takes f = 0..3
#pragma unroll
  for (int sg = 0; sg < 2; sg++)
#pragma unroll
    for (int gg = 0; gg < 4; gg++) x.s[e2(c2 + 4 * sg, f0, gg)] = t[sg][gg];
  wave_sync();
#pragma unroll
  for (int sg = 0; sg < 2; sg++)
#pragma unroll
    for (int f = 0; f < 4; f++) t[sg][f] = x.s[e2(c2 + 4 * sg, f, f0)];
  wave_sync();
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
    dft4s<1>(t[sg]);
#pragma unroll
    for (int h = 0; h < 4; h++) v[4 * sg + h] = t[sg][h];
  }
}

// HORFFT forward of this lane's physical points v (positions as left by
// `inverse`) into one PFP line (element m at dst[lo + ndimr m]).
template <bool FULL>
__device__ __forceinline__ void forward(const Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *__restrict__ dst,
                                        int lo, bool inr, bool live) {
  const int b = x.b, c2 = b >> 2, g0 = b & 3;
  double2 t[2][4];
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
#pragma unroll
    for (int h = 0; h < 4; h++) t[sg][h] = v[4 * sg + h];
    dft4s<-1>(t[sg]);
#pragma unroll
    for (int f = 1; f < 4; f++) t[sg][f] = fz_cmul(t[sg][f], x.t2[4 * g0 + f]);
  }
#pragma unroll
  for (int sg = 0; sg < 2; sg++)
#pragma unroll
    for (int f = 0; f < 4; f++) x.s[e2(c2 + 4 * sg, f, g0)] = t[sg][f];
  wave_sync();
  // lane 4 c2 + f takes g = 0..3
#pragma unroll
  for (int sg = 0; sg < 2; sg++)
#pragma unroll
    for (int gg = 0; gg < 4; gg++) t[sg][gg] = x.s[e2(c2 + 4 * sg, g0, gg)];
  wave_sync();
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
    dft4s<-1>(t[sg]);
#pragma unroll
    for (int e = 0; e < 4; e++) x.s[e1(c2 + 4 * sg, 4 * e + g0)] = t[sg][e];
  }
  wave_sync();
  double2 u[8];
#pragma unroll
  for (int c = 0; c < 8; c++) u[c] = x.s[e1(c, b)];
  wave_sync();
#pragma unroll
  for (int c = 1; c < 8; c++) u[c] = fz_cmul(u[c], x.t1[16 * c + b]);
  dft8s<-1>(u);
  // u[a] = Y[16 a + b]; Y[N - m] sits in lane (16 - b) mod 16 at a' = 7 - a
  // (lane 0: a' = (8 - a) mod 8)
  const double den = (double)(2 * N);
  const int src = (16 - b) & 15;
#pragma unroll
  for (int a = 0; a < (FULL ? 8 : 3); a++) {
    if (16 * a >= g.ntchopdim) break;
    const int m = 16 * a + b;
    double2 pc;
    pc.x = __shfl(u[7 - a].x, src, 16);
    pc.y = __shfl(u[7 - a].y, src, 16);
    if (b == 0) pc = u[(8 - a) & 7];
    if (m < g.ntchopdim && inr) {
      double2 zm = u[a], zc = fz_conj(pc);
      double2 e = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
      double2 d = make_double2(zm.x - zc.x, zm.y - zc.y);
      double2 wd = fz_cmul(x.th[m], d);
      double2 o = make_double2(e.x + 0.5 * wd.y, e.y - 0.5 * wd.x);
      o = make_double2(o.x / den, o.y / den);
      if (m == 0) o.y = 0.0;
      if (m >= g.ntchop || !live) o = make_double2(0.0, 0.0);
      dst[lo + g.ndimr * m] = o;
    }
  }
}

}  // namespace w128

// ---------------------------------------------------------------------------
// NTH = 64: 8 lanes own one theta line (eight lines per wave), each keeping
// 8 of its 64 points.  The 64-point transform is 8 x 8 with one exchange:
//   j = 8 a + b (lane b holds a = 0..7) -> 8-point DFT over a, twiddle
//   exchange: lane c holds b = 0..7     -> 8-point DFT over b
// so lane c ends with the points k = c + 8 d, d = 0..7.
// ---------------------------------------------------------------------------
namespace w64 {

constexpr int N = 64;
constexpr int LP = 72;      // LDS double2 per line (rows of 9 against bank conflicts)
constexpr int MMAX24 = 24;  // NTCHOPDIM bound: slots a = 3, 4 hold no mode
__device__ __forceinline__ int e1(int c, int b) { return c * 9 + b; }
using w256::cj;
using w256::Ctx;  // t1[8 c + b] = W_N^{b c}, th[k] = exp(-i pi k / N)
using w256::dft8s;
using w256::merge_full;
using w256::dft8s_z34;
using w256::wave_sync;

template <bool FULL>
__device__ __forceinline__ void inverse(const Ctx &x, const KGrid &g, const double2 *__restrict__ src, int lo,
                                        bool live, double2 (&v)[8]) {
  const int b = x.b, mmax = g.ntchopdim;
  auto X = [&](int m, bool use) -> double2 {
    use = use && live && m < g.ntchop;
    double2 t = src[lo + (use ? g.ndimr * m : 0)];
    if (!use) t = make_double2(0.0, 0.0);
    if (m == 0) t.y = 0.0;
    return t;
  };
#pragma unroll
  for (int a = 0; a < 8; a++) {
    if (!FULL && (a == 3 || a == 4)) {
      v[a] = make_double2(0.0, 0.0);
      continue;
    }
    const int j = 8 * a + b, jc = N - j;
    if constexpr (FULL) {
      v[a] = merge_full(X(j, j < mmax), fz_conj(X(jc, j > 0 && jc < mmax)), x.th[j]);
      continue;
    }
    const double2 t = x.th[a < 3 ? j : jc];
    const double2 xv = a < 3 ? X(j, j < mmax) : fz_conj(X(jc, jc < mmax));
    const double2 q = a < 3 ? make_double2(1.0 + t.y, t.x) : make_double2(1.0 - t.y, t.x);
    v[a] = fz_cmul(xv, q);
  }
  if constexpr (FULL) dft8s<1>(v);
  else dft8s_z34<1>(v);
#pragma unroll
  for (int c = 1; c < 8; c++) v[c] = fz_cmul(v[c], cj(x.t1[8 * c + b], true));
#pragma unroll
  for (int c = 0; c < 8; c++) x.s[e1(c, b)] = v[c];
  wave_sync();
#pragma unroll
  for (int bb = 0; bb < 8; bb++) v[bb] = x.s[e1(b, bb)];
  wave_sync();
  dft8s<1>(v);
}

template <bool FULL>
__device__ __forceinline__ void forward(const Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *__restrict__ dst,
                                        int lo, bool inr, bool live) {
  const int b = x.b;
  double2 u[8];
#pragma unroll
  for (int d = 0; d < 8; d++) u[d] = v[d];
  dft8s<-1>(u);
#pragma unroll
  for (int bb = 0; bb < 8; bb++) x.s[e1(b, bb)] = u[bb];
  wave_sync();
#pragma unroll
  for (int c = 0; c < 8; c++) u[c] = x.s[e1(c, b)];
  wave_sync();
#pragma unroll
  for (int c = 1; c < 8; c++) u[c] = fz_cmul(u[c], x.t1[8 * c + b]);
  dft8s<-1>(u);
  // u[a] = Y[8 a + b]; Y[N - m] sits in lane (8 - b) mod 8 at a' = 7 - a
  // (lane 0: a' = (8 - a) mod 8)
  const double den = (double)(2 * N);
  const int src = (8 - b) & 7;
#pragma unroll
  for (int a = 0; a < (FULL ? 8 : 3); a++) {
    if (8 * a >= g.ntchopdim) break;
    const int m = 8 * a + b;
    double2 pc;
    pc.x = __shfl(u[7 - a].x, src, 8);
    pc.y = __shfl(u[7 - a].y, src, 8);
    if (b == 0) pc = u[(8 - a) & 7];
    if (m < g.ntchopdim && inr) {
      double2 zm = u[a], zc = fz_conj(pc);
      double2 e = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
      double2 d = make_double2(zm.x - zc.x, zm.y - zc.y);
      double2 wd = fz_cmul(x.th[m], d);
      double2 o = make_double2(e.x + 0.5 * wd.y, e.y - 0.5 * wd.x);
      o = make_double2(o.x / den, o.y / den);
      if (m == 0) o.y = 0.0;
      if (m >= g.ntchop || !live) o = make_double2(0.0, 0.0);
      dst[lo + g.ndimr * m] = o;
    }
  }
}

}  // namespace w64

// ---------------------------------------------------------------------------
// NTH = 32: 4 lanes own one theta line (sixteen lines per wave), each keeping
// 8 of its 32 points.  The 32-point transform is 8 x 4 with one exchange:
//   j = 4 a + b (lane b holds a = 0..7)          -> 8-point DFT over a, twiddle
//   exchange: lane L holds b = 0..3 of c = L, L + 4 -> 4-point DFTs over b
// so lane L ends with the points k = c + 8 d, c = L, L + 4, d = 0..3.
// ---------------------------------------------------------------------------
namespace w32 {

constexpr int N = 32;
constexpr int LP = 40;      // LDS double2 per line (rows of 5 against bank conflicts)
constexpr int MMAX12 = 12;  // NTCHOPDIM bound: slots a = 3, 4 hold no mode
__device__ __forceinline__ int e1(int c, int b) { return c * 5 + b; }
using w256::cj;
using w256::Ctx;  // t1[4 c + b] = W_N^{b c}, th[k] = exp(-i pi k / N)
using w256::dft4s;
using w256::dft8s;
using w256::merge_full;
using w256::dft8s_z34;
using w256::wave_sync;

template <bool FULL>
__device__ __forceinline__ void inverse(const Ctx &x, const KGrid &g, const double2 *__restrict__ src, int lo,
                                        bool live, double2 (&v)[8]) {
  const int b = x.b, mmax = g.ntchopdim;
  auto X = [&](int m, bool use) -> double2 {
    use = use && live && m < g.ntchop;
    double2 t = src[lo + (use ? g.ndimr * m : 0)];
    if (!use) t = make_double2(0.0, 0.0);
    if (m == 0) t.y = 0.0;
    return t;
  };
#pragma unroll
  for (int a = 0; a < 8; a++) {
    if (!FULL && (a == 3 || a == 4)) {
      v[a] = make_double2(0.0, 0.0);
      continue;
    }
    const int j = 4 * a + b, jc = N - j;
    if constexpr (FULL) {
      v[a] = merge_full(X(j, j < mmax), fz_conj(X(jc, j > 0 && jc < mmax)), x.th[j]);
      continue;
    }
    const double2 t = x.th[a < 3 ? j : jc];
    const double2 xv = a < 3 ? X(j, j < mmax) : fz_conj(X(jc, jc < mmax));
    const double2 q = a < 3 ? make_double2(1.0 + t.y, t.x) : make_double2(1.0 - t.y, t.x);
    v[a] = fz_cmul(xv, q);
  }
  if constexpr (FULL) dft8s<1>(v);
  else dft8s_z34<1>(v);
#pragma unroll
  for (int c = 1; c < 8; c++) v[c] = fz_cmul(v[c], cj(x.t1[4 * c + b], true));
#pragma unroll
  for (int c = 0; c < 8; c++) x.s[e1(c, b)] = v[c];
  wave_sync();
  double2 t[2][4];
#pragma unroll
  for (int sg = 0; sg < 2; sg++)
#pragma unroll
    for (int bb = 0; bb < 4; bb++) t[sg][bb] = x.s[e1(b + 4 * sg, bb)];
  wave_sync();
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
    dft4s<1>(t[sg]);
#pragma unroll
    for (int d = 0; d < 4; d++) v[4 * sg + d] = t[sg][d];
  }
}

template <bool FULL>
__device__ __forceinline__ void forward(const Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *__restrict__ dst,
                                        int lo, bool inr, bool live) {
  const int b = x.b;
  double2 t[2][4];
#pragma unroll
  for (int sg = 0; sg < 2; sg++) {
#pragma unroll
    for (int d = 0; d < 4; d++) t[sg][d] = v[4 * sg + d];
    dft4s<-1>(t[sg]);
#pragma unroll
    for (int bb = 0; bb < 4; bb++) x.s[e1(b + 4 * sg, bb)] = t[sg][bb];
  }
  wave_sync();
  double2 u[8];
#pragma unroll
  for (int c = 0; c < 8; c++) u[c] = x.s[e1(c, b)];
  wave_sync();
#pragma unroll
  for (int c = 1; c < 8; c++) u[c] = fz_cmul(u[c], x.t1[4 * c + b]);
  dft8s<-1>(u);
  // u[a] = Y[4 a + b]; Y[N - m] sits in lane (4 - b) mod 4 at a' = 7 - a
  // (lane 0: a' = (8 - a) mod 8)
  const double den = (double)(2 * N);
  const int src = (4 - b) & 3;
#pragma unroll
  for (int a = 0; a < (FULL ? 8 : 3); a++) {
    if (4 * a >= g.ntchopdim) break;
    const int m = 4 * a + b;
    double2 pc;
    pc.x = __shfl(u[7 - a].x, src, 4);
    pc.y = __shfl(u[7 - a].y, src, 4);
    if (b == 0) pc = u[(8 - a) & 7];
    if (m < g.ntchopdim && inr) {
      double2 zm = u[a], zc = fz_conj(pc);
      double2 e = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
      double2 d = make_double2(zm.x - zc.x, zm.y - zc.y);
      double2 wd = fz_cmul(x.th[m], d);
      double2 o = make_double2(e.x + 0.5 * wd.y, e.y - 0.5 * wd.x);
      o = make_double2(o.x / den, o.y / den);
      if (m == 0) o.y = 0.0;
      if (m >= g.ntchop || !live) o = make_double2(0.0, 0.0);
      dst[lo + g.ndimr * m] = o;
    }
  }
}

}  // namespace w32

// ---------------------------------------------------------------------------
// NTH = 512: a wave owns one theta line, each lane 8 of its points; eight
// waves, and eight adjacent radial nodes, a block.  The 512-point transform is
// 8 x 8 x 8:
//   j = 64 a + b (lane b holds a = 0..7)          -> 8-point DFT over a, twiddle
//   exchange: lane 8 c + f (b = 8 e + f) holds e = 0..7 of c
//                                                  -> 8-point DFT over e, twiddle
//   exchange: lane 8 c + g holds f = 0..7          -> 8-point DFT over f
// so lane 8 c + g ends with the points k = c + 8 g + 64 h, h = 0..7.
// ---------------------------------------------------------------------------
namespace w512 {

constexpr int N = 512;
constexpr int LP = 576;       // LDS double2 per line (rows of 9 against bank conflicts)
constexpr int MMAX192 = 192;  // NTCHOPDIM bound without FULL: slots a = 3, 4 hold no mode
__device__ __forceinline__ int e1(int c, int b) { return c * 72 + b; }
__device__ __forceinline__ int e2(int c, int f, int g) { return c * 72 + f * 9 + g; }
using w256::cj;
using w256::Ctx;  // t1[64 c + b] = W_N^{b c}, t2[8 g + f] = W_N^{8 f g}, th[k] = exp(-i pi k / N)
using w256::dft8s;
using w256::dft8s_z34;
using w256::merge_full;
using w256::wave_sync;

template <bool FULL>
__device__ __forceinline__ void inverse(const Ctx &x, const KGrid &g, const double2 *__restrict__ src, int lo,
                                        bool live, double2 (&v)[8]) {
  const int b = x.b, mmax = g.ntchopdim;
  auto X = [&](int m, bool use) -> double2 {
    use = use && live && m < g.ntchop;
    double2 t = src[lo + (use ? g.ndimr * m : 0)];
    if (!use) t = make_double2(0.0, 0.0);
    if (m == 0) t.y = 0.0;
    return t;
  };
#pragma unroll
  for (int a = 0; a < 8; a++) {
    if (!FULL && (a == 3 || a == 4)) {
      v[a] = make_double2(0.0, 0.0);
      continue;
    }
    const int j = 64 * a + b, jc = N - j;
    if constexpr (FULL) {
      v[a] = merge_full(X(j, j < mmax), fz_conj(X(jc, j > 0 && jc < mmax)), x.th[j]);
      continue;
    }
    const double2 t = x.th[a < 3 ? j : jc];
    const double2 xv = a < 3 ? X(j, j < mmax) : fz_conj(X(jc, jc < mmax));
    const double2 q = a < 3 ? make_double2(1.0 + t.y, t.x) : make_double2(1.0 - t.y, t.x);
    v[a] = fz_cmul(xv, q);
  }
  if constexpr (FULL) dft8s<1>(v);
  else dft8s_z34<1>(v);
#pragma unroll
  for (int c = 1; c < 8; c++) v[c] = fz_cmul(v[c], cj(x.t1[64 * c + b], true));
#pragma unroll
  for (int c = 0; c < 8; c++) x.s[e1(c, b)] = v[c];
  wave_sync();
  const int c0 = b >> 3, f0 = b & 7;
#pragma unroll
  for (int e = 0; e < 8; e++) v[e] = x.s[e1(c0, 8 * e + f0)];
  wave_sync();
  dft8s<1>(v);
#pragma unroll
  for (int gg = 1; gg < 8; gg++) v[gg] = fz_cmul(v[gg], cj(x.t2[8 * gg + f0], true));
#pragma unroll
  for (int gg = 0; gg < 8; gg++) x.s[e2(c0, f0, gg)] = v[gg];
  wave_sync();
#pragma unroll
  for (int f = 0; f < 8; f++) v[f] = x.s[e2(c0, f, f0)];
  wave_sync();
  dft8s<1>(v);
}

template <bool FULL>
__device__ __forceinline__ void forward(const Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *__restrict__ dst,
                                        int lo, bool inr, bool live) {
  const int b = x.b, c0 = b >> 3, f0 = b & 7;
  double2 u[8];
#pragma unroll
  for (int h = 0; h < 8; h++) u[h] = v[h];
  dft8s<-1>(u);
#pragma unroll
  for (int f = 1; f < 8; f++) u[f] = fz_cmul(u[f], x.t2[8 * f0 + f]);
#pragma unroll
  for (int f = 0; f < 8; f++) x.s[e2(c0, f, f0)] = u[f];
  wave_sync();
#pragma unroll
  for (int gg = 0; gg < 8; gg++) u[gg] = x.s[e2(c0, f0, gg)];
  wave_sync();
  dft8s<-1>(u);
#pragma unroll
  for (int e = 0; e < 8; e++) x.s[e1(c0, 8 * e + f0)] = u[e];
  wave_sync();
#pragma unroll
  for (int c = 0; c < 8; c++) u[c] = x.s[e1(c, b)];
  wave_sync();
#pragma unroll
  for (int c = 1; c < 8; c++) u[c] = fz_cmul(u[c], x.t1[64 * c + b]);
  dft8s<-1>(u);
  // u[a] = Y[64 a + b]; Y[N - m] sits in lane (64 - b) mod 64 at a' = 7 - a
  // (lane 0: a' = (8 - a) mod 8)
  const double den = (double)(2 * N);
  const int src = (64 - b) & 63;
#pragma unroll
  for (int a = 0; a < (FULL ? 8 : 3); a++) {
    if (64 * a >= g.ntchopdim) break;
    const int m = 64 * a + b;
    double2 pc;
    pc.x = __shfl(u[7 - a].x, src, 64);
    pc.y = __shfl(u[7 - a].y, src, 64);
    if (b == 0) pc = u[(8 - a) & 7];
    if (m < g.ntchopdim && inr) {
      double2 zm = u[a], zc = fz_conj(pc);
      double2 e = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
      double2 d = make_double2(zm.x - zc.x, zm.y - zc.y);
      double2 wd = fz_cmul(x.th[m], d);
      double2 o = make_double2(e.x + 0.5 * wd.y, e.y - 0.5 * wd.x);
      o = make_double2(o.x / den, o.y / den);
      if (m == 0) o.y = 0.0;
      if (m >= g.ntchop || !live) o = make_double2(0.0, 0.0);
      dst[lo + g.ndimr * m] = o;
    }
  }
}

}  // namespace w512

// ---------------------------------------------------------------------------
// NTH = 16: 2 lanes own one theta line (32 lines per wave), each keeping 8 of
// its points, with a 8 x 2 transform: j = 2 a + b (lane b holds a = 0..7) ->
// 8-point DFT over a, twiddle, 2-point DFT between the two lanes; lane b ends
// with the points k = c + 8 b.  No LDS.
// ---------------------------------------------------------------------------
namespace w16 {

constexpr int N = 16;
constexpr int MMAX6 = 6;  // NTCHOPDIM bound without FULL: slots a = 3, 4 hold no mode
using w256::cj;
using w256::Ctx;  // t1[2 c + b] = W_N^{b c}, th[k] = exp(-i pi k / N)
using w256::dft8s;
using w256::dft8s_z34;
using w256::merge_full;

// v[c] = v0[c] + v1[c] in lane 0, v0[c] - v1[c] in lane 1
__device__ __forceinline__ void pair2(int b, double2 (&v)[8]) {
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const double ox = __shfl_xor(v[c].x, 1, 64), oy = __shfl_xor(v[c].y, 1, 64);
    v[c] = b ? make_double2(ox - v[c].x, oy - v[c].y) : make_double2(v[c].x + ox, v[c].y + oy);
  }
}

template <bool FULL>
__device__ __forceinline__ void inverse(const Ctx &x, const KGrid &g, const double2 *__restrict__ src, int lo,
                                        bool live, double2 (&v)[8]) {
  const int b = x.b, mmax = g.ntchopdim;
  auto X = [&](int m, bool use) -> double2 {
    use = use && live && m < g.ntchop;
    double2 t = src[lo + (use ? g.ndimr * m : 0)];
    if (!use) t = make_double2(0.0, 0.0);
    if (m == 0) t.y = 0.0;
    return t;
  };
#pragma unroll
  for (int a = 0; a < 8; a++) {
    if (!FULL && (a == 3 || a == 4)) {
      v[a] = make_double2(0.0, 0.0);
      continue;
    }
    const int j = 2 * a + b, jc = N - j;
    if constexpr (FULL) {
      v[a] = merge_full(X(j, j < mmax), fz_conj(X(jc, j > 0 && jc < mmax)), x.th[j]);
      continue;
    }
    const double2 t = x.th[a < 3 ? j : jc];
    const double2 xv = a < 3 ? X(j, j < mmax) : fz_conj(X(jc, jc < mmax));
    const double2 q = a < 3 ? make_double2(1.0 + t.y, t.x) : make_double2(1.0 - t.y, t.x);
    v[a] = fz_cmul(xv, q);
  }
  if constexpr (FULL) dft8s<1>(v);
  else dft8s_z34<1>(v);
#pragma unroll
  for (int c = 1; c < 8; c++) v[c] = fz_cmul(v[c], cj(x.t1[2 * c + b], true));
  pair2(b, v);
}

template <bool FULL>
__device__ __forceinline__ void forward(const Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *__restrict__ dst,
                                        int lo, bool inr, bool live) {
  const int b = x.b;
  double2 u[8];
#pragma unroll
  for (int c = 0; c < 8; c++) u[c] = v[c];
  pair2(b, u);
#pragma unroll
  for (int c = 1; c < 8; c++) u[c] = fz_cmul(u[c], x.t1[2 * c + b]);
  dft8s<-1>(u);
  // u[a] = Y[2 a + b]; Y[N - m] is this lane's a' = (8 - a) mod 8 (b = 0), 7 - a (b = 1)
  const double den = (double)(2 * N);
#pragma unroll
  for (int a = 0; a < (FULL ? 8 : 3); a++) {
    const int m = 2 * a + b;
    const double2 pc = b ? u[7 - a] : u[(8 - a) & 7];
    if (m < g.ntchopdim && inr) {
      double2 zm = u[a], zc = fz_conj(pc);
      double2 e = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
      double2 d = make_double2(zm.x - zc.x, zm.y - zc.y);
      double2 wd = fz_cmul(x.th[m], d);
      double2 o = make_double2(e.x + 0.5 * wd.y, e.y - 0.5 * wd.x);
      o = make_double2(o.x / den, o.y / den);
      if (m == 0) o.y = 0.0;
      if (m >= g.ntchop || !live) o = make_double2(0.0, 0.0);
      dst[lo + g.ndimr * m] = o;
    }
  }
}

}  // namespace w16

// ---------------------------------------------------------------------------
// NTH = N = 2, 4, 8: a lane owns a theta line, its points in the first N of
// the 8 slots.
// ---------------------------------------------------------------------------
template <int N>
struct w8 {
  template <int S>
  __device__ __forceinline__ static void dft(double2 (&v)[8]) {
    if constexpr (N == 8) {
      w256::dft8s<S>(v);
    } else if constexpr (N == 4) {
      double2 y[4] = {v[0], v[1], v[2], v[3]};
      w256::dft4s<S>(y);
#pragma unroll
      for (int k = 0; k < 4; k++) v[k] = y[k];
    } else {
      const double2 a = v[0], b = v[1];
      v[0] = w256::cadd(a, b);
      v[1] = w256::csub(a, b);
    }
  }
  __device__ __forceinline__ static void inverse(const w256::Ctx &x, const KGrid &g, const double2 *__restrict__ src, int lo,
                                                 bool live, double2 (&v)[8]) {
    const int mmax = g.ntchopdim;
    auto X = [&](int m, bool use) -> double2 {
      use = use && live && m < g.ntchop;
      double2 t = src[lo + (use ? g.ndimr * m : 0)];
      if (!use) t = make_double2(0.0, 0.0);
      if (m == 0) t.y = 0.0;
      return t;
    };
#pragma unroll
    for (int j = 0; j < 8; j++)
      v[j] = j < N ? w256::merge_full(X(j, j < mmax), fz_conj(X(N - j, j > 0 && N - j < mmax)), x.th[j < N ? j : 0])
                   : make_double2(0.0, 0.0);
    dft<1>(v);
  }
  __device__ __forceinline__ static void forward(const w256::Ctx &x, const KGrid &g, const double2 (&v)[8],
                                                 double2 *__restrict__ dst, int lo, bool inr, bool live) {
    double2 u[8];
#pragma unroll
    for (int c = 0; c < 8; c++) u[c] = v[c];
    dft<-1>(u);
    const double den = (double)(2 * N);
#pragma unroll
    for (int m = 0; m < N; m++) {
      if (m < g.ntchopdim && inr) {
        double2 zm = u[m], zc = fz_conj(u[(N - m) % N]);
        double2 e = make_double2(0.5 * (zm.x + zc.x), 0.5 * (zm.y + zc.y));
        double2 d = make_double2(zm.x - zc.x, zm.y - zc.y);
        double2 wd = fz_cmul(x.th[m], d);
        double2 o = make_double2(e.x + 0.5 * wd.y, e.y - 0.5 * wd.x);
        o = make_double2(o.x / den, o.y / den);
        if (m == 0) o.y = 0.0;
        if (m >= g.ntchop || !live) o = make_double2(0.0, 0.0);
        dst[lo + g.ndimr * m] = o;
      }
    }
  }
};

// Line shapes of the kernels below: lanes per theta line,
// LDS per line, the NTCHOPDIM bound of the pruned first stage, and the
// per-lane twiddle tables (T1[LANES c + b] = W_N^{b c}; T2 of NTH = 128's
// middle stage, T2[4 g + f] = W_N^{8 f g}).
template <int NN>
struct LineTiny {
  static constexpr int N = NN, LANES = 1, LP = 8, MMAX = 0, NT2 = 1;
  __device__ static void tables(int, double2 *, double2 *, const double2 *) {}
  template <bool FULL>
  __device__ static void inverse(const w256::Ctx &x, const KGrid &g, const double2 *src, int lo, bool live,
                                 double2 (&v)[8]) {
    w8<N>::inverse(x, g, src, lo, live, v);
  }
  template <bool FULL>
  __device__ static void forward(const w256::Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *dst, int lo, bool inr,
                                 bool live) {
    w8<N>::forward(x, g, v, dst, lo, inr, live);
  }
};
struct Line16 {
  static constexpr int N = 16, LANES = 2, THREADS = 256, LP = 16, MMAX = w16::MMAX6, NT2 = 1;
  // theta index of the point in slot i of lane b
  __device__ static int point(int b, int i) { return i + 8 * b; }
  __device__ static void tables(int q, double2 *T1, double2 *, const double2 *tw) {
    if (q < 16) T1[q] = tw[(q & 1) * (q >> 1)];
  }
  template <bool FULL>
  __device__ static void inverse(const w256::Ctx &x, const KGrid &g, const double2 *src, int lo, bool live,
                                 double2 (&v)[8]) {
    w16::inverse<FULL>(x, g, src, lo, live, v);
  }
  template <bool FULL>
  __device__ static void forward(const w256::Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *dst, int lo, bool inr,
                                 bool live) {
    w16::forward<FULL>(x, g, v, dst, lo, inr, live);
  }
};
struct Line128 {
  static constexpr int N = 128, LANES = 16, THREADS = 256, LP = w128::LP, MMAX = w128::MMAX48, NT2 = 16;
  // theta index of the point in slot i of lane b
  __device__ static int point(int b, int i) { return ((b >> 2) + 4 * (i >> 2)) + 8 * (b & 3) + 32 * (i & 3); }
  __device__ static void tables(int q, double2 *T1, double2 *T2, const double2 *tw) {
    if (q < 128) T1[q] = tw[(q & 15) * (q >> 4)];
    if (q < 16) T2[q] = tw[8 * (q & 3) * (q >> 2)];
  }
  template <bool FULL>
  __device__ static void inverse(const w256::Ctx &x, const KGrid &g, const double2 *src, int lo, bool live,
                                 double2 (&v)[8]) {
    w128::inverse<FULL>(x, g, src, lo, live, v);
  }
  template <bool FULL>
  __device__ static void forward(const w256::Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *dst, int lo, bool inr,
                                 bool live) {
    w128::forward<FULL>(x, g, v, dst, lo, inr, live);
  }
};
struct Line32 {
  static constexpr int N = 32, LANES = 4, THREADS = 256, LP = w32::LP, MMAX = w32::MMAX12, NT2 = 1;
  // theta index of the point in slot i of lane b
  __device__ static int point(int b, int i) { return (b + 4 * (i >> 2)) + 8 * (i & 3); }
  __device__ static void tables(int q, double2 *T1, double2 *, const double2 *tw) {
    if (q < 32) T1[q] = tw[(q & 3) * (q >> 2)];
  }
  template <bool FULL>
  __device__ static void inverse(const w256::Ctx &x, const KGrid &g, const double2 *src, int lo, bool live,
                                 double2 (&v)[8]) {
    w32::inverse<FULL>(x, g, src, lo, live, v);
  }
  template <bool FULL>
  __device__ static void forward(const w256::Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *dst, int lo, bool inr,
                                 bool live) {
    w32::forward<FULL>(x, g, v, dst, lo, inr, live);
  }
};
struct Line64 {
  static constexpr int N = 64, LANES = 8, THREADS = 256, LP = w64::LP, MMAX = w64::MMAX24, NT2 = 1;
  // theta index of the point in slot i of lane b
  __device__ static int point(int b, int i) { return b + 8 * i; }
  __device__ static void tables(int q, double2 *T1, double2 *, const double2 *tw) {
    if (q < 64) T1[q] = tw[(q & 7) * (q >> 3)];
  }
  template <bool FULL>
  __device__ static void inverse(const w256::Ctx &x, const KGrid &g, const double2 *src, int lo, bool live,
                                 double2 (&v)[8]) {
    w64::inverse<FULL>(x, g, src, lo, live, v);
  }
  template <bool FULL>
  __device__ static void forward(const w256::Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *dst, int lo, bool inr,
                                 bool live) {
    w64::forward<FULL>(x, g, v, dst, lo, inr, live);
  }
};

struct Line512 {
  static constexpr int N = 512, LANES = 64, THREADS = 512, LP = w512::LP, MMAX = w512::MMAX192, NT2 = 64;
  // theta index of the point in slot i of lane b
  __device__ static int point(int b, int i) { return (b >> 3) + 8 * (b & 7) + 64 * i; }
  __device__ static void tables(int q, double2 *T1, double2 *T2, const double2 *tw) {
    T1[q] = tw[(q & 63) * (q >> 6)];
    if (q < 64) T2[q] = tw[8 * (q & 7) * (q >> 3)];
  }
  template <bool FULL>
  __device__ static void inverse(const w256::Ctx &x, const KGrid &g, const double2 *src, int lo, bool live,
                                 double2 (&v)[8]) {
    w512::inverse<FULL>(x, g, src, lo, live, v);
  }
  template <bool FULL>
  __device__ static void forward(const w256::Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *dst, int lo, bool inr,
                                 bool live) {
    w512::forward<FULL>(x, g, v, dst, lo, inr, live);
  }
};

// The NTH = 256 kernel's products and field order on the lines of NTH = 512
// (Line512: 64 lanes, 8 lines per block of eight waves), NTH = 128
// (Line128: 16 lanes, 16 lines per block), NTH = 64 (Line64: 8 lanes, 32
// lines), NTH = 32 (Line32: 4 lanes, 64 lines) or NTH = 16 (Line16: 2 lanes,
// 128 lines); a block takes adjacent
// radial nodes of one z plane.
template <class L, bool LINEAR, bool FULL = false>
__global__ void __launch_bounds__(L::THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_fused_products_reg(KGrid g, const double *__restrict__ rsq, const double2 *tw, const double2 *twh, FusedIO io,
                     double two_omega, double n2) {
  if (blockIdx.x == 0 && threadIdx.x == 0 && io.zl) io.zl[0] = 0.0;
  constexpr int N = L::N, LANES = L::LANES, LINES = L::THREADS / LANES;
  __shared__ double2 S[LINES * L::LP];
  __shared__ double2 Y[LINES * N];  // [line][point i][lane]
  __shared__ double2 T1[N], T2[L::NT2], TH[N + 1];
  const int nrb = (g.ndimr + LINES - 1) / LINES;
  const int lid = xcd_logical(nrb * g.ndimx);
  if (lid < 0) return;
  {
    const int q = threadIdx.x;
    L::tables(q, T1, T2, tw);
    if (q <= N) TH[q] = twh[q];
    if (L::THREADS == N && q == 0) TH[N] = twh[N];
  }
  __syncthreads();
  const int z = lid / nrb, line = threadIdx.x / LANES;
  const int rr = (lid % nrb) * LINES + line;
  const bool inr = rr < g.ndimr, live = rr < g.nr;
  w256::Ctx x;
  x.t1 = T1;
  x.t2 = T2;
  x.th = TH;
  x.s = S + line * L::LP;
  x.b = threadIdx.x % LANES;
  double2 *ys = Y + line * N + x.b;
  const size_t off = (size_t)(rr - line) + (size_t)g.ndimr * g.ndimth * z;  // same for the block
  const int lo = inr ? line : 0;
  auto in = [&](int q) { return io.in[q] + off; };
  auto out = [&](int q) { return io.out[q] + off; };
  const double r2 = live ? rsq[rr] : 1.0;

  double2 A[8], B[8], C[8], U[8], V[8], T[8];
  L::template inverse<FULL>(x, g, in(0), lo, live, A);  // rur
  L::template inverse<FULL>(x, g, in(1), lo, live, B);  // rup
  L::template inverse<FULL>(x, g, in(2), lo, live, C);  // uz
  // oz: U = rup oz, V = rur oz
  L::template inverse<FULL>(x, g, in(5), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    U[i] = make_double2(B[i].x * T[i].x, B[i].y * T[i].y);
    V[i] = make_double2(A[i].x * T[i].x, A[i].y * T[i].y);
  }
  // ror: Y = uz ror - rur oz (to LDS); V = rup ror
  L::template inverse<FULL>(x, g, in(3), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    ys[LANES * i] = make_double2(C[i].x * T[i].x - V[i].x, C[i].y * T[i].y - V[i].y);
    V[i] = make_double2(B[i].x * T[i].x, B[i].y * T[i].y);
  }
  // rop: X = rup oz - uz rop in U; Z = (rur rop - rup ror) / r^2 in V
  L::template inverse<FULL>(x, g, in(4), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    U[i] = make_double2(U[i].x - C[i].x * T[i].x, U[i].y - C[i].y * T[i].y);
    V[i] = make_double2((A[i].x * T[i].x - V[i].x) / r2, (A[i].y * T[i].y - V[i].y) / r2);
  }
  // ror, rop, oz are read: the outputs may now overwrite them
  if (LINEAR) {
#pragma unroll
    for (int i = 0; i < 8; i++) U[i] = make_double2(U[i].x + two_omega * B[i].x, U[i].y + two_omega * B[i].y);
  }
  L::template forward<FULL>(x, g, U, out(0), lo, inr, live);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    T[i] = ys[LANES * i];
    if (LINEAR) T[i] = make_double2(T[i].x - two_omega * A[i].x, T[i].y - two_omega * A[i].y);
  }
  L::template forward<FULL>(x, g, T, out(1), lo, inr, live);
  if (LINEAR) {
    // W: N_z = Z - W
    L::template inverse<FULL>(x, g, in(9), lo, live, T);
#pragma unroll
    for (int i = 0; i < 8; i++) V[i] = make_double2(V[i].x - T[i].x, V[i].y - T[i].y);
  }
  L::template forward<FULL>(x, g, V, out(2), lo, inr, live);
  // rbr, rbp: A = rur rbr + rup rbp
  L::template inverse<FULL>(x, g, in(6), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) A[i] = make_double2(A[i].x * T[i].x, A[i].y * T[i].y);
  L::template inverse<FULL>(x, g, in(7), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) A[i] = make_double2(A[i].x + B[i].x * T[i].x, A[i].y + B[i].y * T[i].y);
  // bz: N_b = -(T / r^2 + uz bz) (+ Nbar^2 uz)
  L::template inverse<FULL>(x, g, in(8), lo, live, T);
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const double vr = A[i].x / r2 + C[i].x * T[i].x, vi = A[i].y / r2 + C[i].y * T[i].y;
    double2 nb = make_double2(-vr, -vi);
    if (LINEAR) nb = make_double2(nb.x + n2 * C[i].x, nb.y + n2 * C[i].y);
    A[i] = nb;
  }
  L::template forward<FULL>(x, g, A, out(3), lo, inr, live);
}

struct Line256 {
  static constexpr int N = 256, LANES = 32, THREADS = 256, LP = w256::LP, MMAX = w256::MMAX96, NT2 = 32;
  // theta index of the point in slot i of lane b
  __device__ static int point(int b, int i) { return (b >> 2) + 8 * ((b & 3) + 4 * (i >> 2)) + 64 * (i & 3); }
  __device__ static void tables(int q, double2 *T1, double2 *T2, const double2 *tw) {
    if (q < 256) T1[q] = tw[(q & 31) * (q >> 5)];
    if (q < 32) T2[q] = tw[8 * (q & 3) * (q >> 2)];
  }
  template <bool FULL>
  __device__ static void inverse(const w256::Ctx &x, const KGrid &g, const double2 *src, int lo, bool live,
                                 double2 (&v)[8]) {
    w256::inverse<FULL>(x, g, src, lo, live, v);
  }
  template <bool FULL>
  __device__ static void forward(const w256::Ctx &x, const KGrid &g, const double2 (&v)[8], double2 *dst, int lo, bool inr,
                                 bool live) {
    w256::forward<FULL>(x, g, v, dst, lo, inr, live);
  }
};

// Small grids: the register kernels' lines, a wave a field.  Each wave takes
// its field of the block's 64 / LANES lines to physical space and leaves the
// points in LDS, where the first four waves form one product each, at the
// same points as their lanes' own, and transform it forward.  The ten inverse
// and four forward transforms that a line of the register kernels runs one
// after the other are here one of each, in return for a fourth of the work
// per wave.
template <class L, bool LINEAR, bool FULL>
__global__ void __launch_bounds__(LINEAR ? 640 : 576)
k_fused_products_wide(KGrid g, const double *__restrict__ rsq, const double2 *tw, const double2 *twh, FusedIO io,
                      double two_omega, double n2) {
  if (blockIdx.x == 0 && threadIdx.x == 0 && io.zl) io.zl[0] = 0.0;
  constexpr int N = L::N, LANES = L::LANES, LINES = 64 / LANES, NF = LINEAR ? 10 : 9;
  constexpr int SL = LINES * L::LP;  // >= 512: the exchanges of a wave, then its 8 points a lane
  static_assert(SL >= 512, "a field's points");
  __shared__ double2 S[NF * SL];
  __shared__ double2 T1[N], T2[L::NT2], TH[N + 1];
  const int nrb = (g.ndimr + LINES - 1) / LINES;
  const int lid = xcd_logical(nrb * g.ndimx);
  if (lid < 0) return;
  {
    const int q = threadIdx.x;
    if (q < 512) L::tables(q, T1, T2, tw);
    if (q <= N) TH[q] = twh[q];
  }
  __syncthreads();
  const int z = lid / nrb, lane = threadIdx.x & 63, line = lane / LANES;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rr = (lid % nrb) * LINES + line;
  const bool inr = rr < g.ndimr, live = rr < g.nr;
  w256::Ctx x;
  x.t1 = T1;
  x.t2 = T2;
  x.th = TH;
  x.s = S + w * SL + line * L::LP;
  x.b = lane % LANES;
  const size_t off = (size_t)(rr - line) + (size_t)g.ndimr * g.ndimth * z;  // same for the block
  const int lo = inr ? line : 0;
  double2 v[8];
  L::template inverse<FULL>(x, g, io.in[w] + off, lo, live, v);
  w256::wave_sync();
#pragma unroll
  for (int i = 0; i < 8; i++) S[w * SL + 64 * i + lane] = v[i];
  __syncthreads();
  auto F = [&](int q, int i) { return S[q * SL + 64 * i + lane]; };
  if (w < 4) {
    const double r2 = live ? rsq[rr] : 1.0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
      if (w == 0) {
        const double2 B = F(1, i), C = F(2, i), E = F(4, i), O = F(5, i);
        v[i] = make_double2(B.x * O.x - C.x * E.x, B.y * O.y - C.y * E.y);
        if (LINEAR) v[i] = make_double2(v[i].x + two_omega * B.x, v[i].y + two_omega * B.y);
      } else if (w == 1) {
        const double2 A = F(0, i), C = F(2, i), D = F(3, i), O = F(5, i);
        v[i] = make_double2(C.x * D.x - A.x * O.x, C.y * D.y - A.y * O.y);
        if (LINEAR) v[i] = make_double2(v[i].x - two_omega * A.x, v[i].y - two_omega * A.y);
      } else if (w == 2) {
        const double2 A = F(0, i), B = F(1, i), D = F(3, i), E = F(4, i);
        v[i] = make_double2((A.x * E.x - B.x * D.x) / r2, (A.y * E.y - B.y * D.y) / r2);
        if (LINEAR) {
          const double2 W = F(9, i);
          v[i] = make_double2(v[i].x - W.x, v[i].y - W.y);
        }
      } else {
        const double2 A = F(0, i), B = F(1, i), C = F(2, i), P = F(6, i), Q = F(7, i), R = F(8, i);
        const double tr = A.x * P.x + B.x * Q.x, ti = A.y * P.y + B.y * Q.y;
        v[i] = make_double2(-(tr / r2 + C.x * R.x), -(ti / r2 + C.y * R.y));
        if (LINEAR) v[i] = make_double2(v[i].x + n2 * C.x, v[i].y + n2 * C.y);
      }
    }
  }
  __syncthreads();
  if (w < 4) L::template forward<FULL>(x, g, v, io.out[w] + off, lo, inr, live);
}

// HORFFT of one field (PFP m < NTCHOPDIM <-> PPP slots, in place) on the same
// lines: a wave transforms whole theta lines without a barrier, and a block
// takes adjacent radial nodes of one plane.  Radial lines are not whole cache
// lines; the blocks that share one run on one XCD.
template <class L, bool FULL, bool FWD>
__global__ void __launch_bounds__(L::THREADS) k_horfft_line(KGrid g, const double2 *tw, const double2 *twh, HorJobs jobs) {
  constexpr int N = L::N, LANES = L::LANES, LINES = L::THREADS / LANES;
  __shared__ double2 S[LINES * L::LP];
  __shared__ double2 T1[N], T2[L::NT2], TH[N + 1];
  const int nrb = (g.ndimr + LINES - 1) / LINES;
  const int lid = xcd_logical(nrb * g.ndimx * jobs.n);
  if (lid < 0) return;
  {
    const int q = threadIdx.x;
    L::tables(q, T1, T2, tw);
    if (q <= N) TH[q] = twh[q];
    if (L::THREADS == N && q == 0) TH[N] = twh[N];
  }
  __syncthreads();
  const int z = lid / nrb % g.ndimx, line = threadIdx.x / LANES;
  const int rr = (lid % nrb) * LINES + line;
  const bool inr = rr < g.ndimr, live = rr < g.nr;
  w256::Ctx x;
  x.t1 = T1;
  x.t2 = T2;
  x.th = TH;
  x.s = S + line * L::LP;
  x.b = threadIdx.x % LANES;
  double2 *a = jobs.a[lid / nrb / g.ndimx] + (size_t)(rr - line) + (size_t)g.ndimr * g.ndimth * z;  // same for the block
  const int lo = inr ? line : 0;
  double2 v[8];
  if constexpr (FWD) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      v[i] = a[lo + g.ndimr * L::point(x.b, i)];
      if (!live) v[i] = make_double2(0.0, 0.0);
    }
    L::template forward<FULL>(x, g, v, a, lo, inr, live);
  } else {
    L::template inverse<FULL>(x, g, a, lo, live, v);
    if (!inr) return;
#pragma unroll
    for (int i = 0; i < 8; i++) a[lo + g.ndimr * L::point(x.b, i)] = live ? v[i] : make_double2(0.0, 0.0);
    if (x.b == 0) a[lo + g.ndimr * N] = make_double2(0.0, 0.0);
  }
}

template <class L, bool FULL>
static void horfft_line(mlg_ctx *c, const KGrid &g, const HorJobs &jobs, bool fwd) {
  constexpr int lines = L::THREADS / L::LANES;
  const dim3 grid(xcd_grid((g.ndimr + lines - 1) / lines * g.ndimx * jobs.n));
  if (fwd)
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_horfft_line<L, FULL, true>), grid, dim3(L::THREADS), 0, c->stream, g, c->d.tw_t,
                       c->d.tw_h, jobs);
  else
    hipLaunchKernelGGL(HIP_KERNEL_NAME(k_horfft_line<L, FULL, false>), grid, dim3(L::THREADS), 0, c->stream, g, c->d.tw_t,
                       c->d.tw_h, jobs);
}
template <class L>
static int horfft_lines(mlg_ctx *c, const HorJobs &jobs, bool fwd) {
  const KGrid g = kgrid(c);
  if (g.ntchopdim <= L::MMAX) horfft_line<L, false>(c, g, jobs, fwd);
  else horfft_line<L, true>(c, g, jobs, fwd);
  MLG_CHECK_HIP(hipGetLastError());
  return 0;
}
int launch_horfft_line(mlg_ctx *c, const HorJobs &jobs, bool fwd) {
  switch (c->g.nth) {
    case 16: return horfft_lines<Line16>(c, jobs, fwd);
    case 32: return horfft_lines<Line32>(c, jobs, fwd);
    case 64: return horfft_lines<Line64>(c, jobs, fwd);
    case 128: return horfft_lines<Line128>(c, jobs, fwd);
    case 256: return horfft_lines<Line256>(c, jobs, fwd);
    case 512: return horfft_lines<Line512>(c, jobs, fwd);
    default: return MLG_E_ARG;
  }
}

bool fused_products_supported(const mlg_ctx *c) {
  return fused_line_length(c->g.nth) || c->fp.n;
}

// One wave a field or a line's fields in one wave.  Truncations past 3/8 of
// NTH (FULL: both terms in the merge) spill in the kernels that hold all
// fields, so they go a wave a field: at 256 x NTH x 256, NTH = 32, 64, 128 163,
// 335, 777 us against 295, 541, 884.  At NTH = 512, where a wave a field is one
// line a block, only up to sixteen blocks a CU: 64 x 512 x 32 (2080 blocks) 129
// us against 147, 128 x 512 x 32 (4128) 265 against 253, 128 x 512 x 64 525
// against 468, 192 x 512 x 384 4.46 ms against 3.75.  Others do while the
// blocks fill the chip at most three times (one block a CU): at NR = 64, NX =
// 32 8.1 us against 20.3 (NTH = 32, 160 blocks), 14.3 against 20.4 (64, 288)
// and 25.2 against 28.8 (128, 544), but 33.6 against 28.5 at 128 x 64 x 64
// (1088) and 234 against 150 at 256 x 64 x 256.
template <class L, bool LINEAR>
static int launch_line(mlg_ctx *c, const FusedIO &io, double two_omega, double n2) {
  KGrid g = kgrid(c);
  constexpr int wl = 64 / L::LANES;
  const int wide = (g.ndimr + wl - 1) / wl * g.ndimx;
#define L_WIDE(FULL_)                                                                                    \
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fused_products_wide<L, LINEAR, FULL_>), dim3(xcd_grid(wide)),     \
                     dim3(LINEAR ? 640 : 576), 0, c->stream, g, c->d.r, c->d.tw_t, c->d.tw_h, io, two_omega, n2)
#define L_REG(FULL_)                                                                                     \
  hipLaunchKernelGGL(HIP_KERNEL_NAME(k_fused_products_reg<L, LINEAR, FULL_>),                            \
                     dim3(xcd_grid((g.ndimr + L::THREADS / L::LANES - 1) / (L::THREADS / L::LANES) * g.ndimx)), \
                     dim3(L::THREADS), 0, c->stream, g, c->d.r, c->d.tw_t, c->d.tw_h, io, two_omega, n2)
  if constexpr (L::N == 512) {
    if (g.ntchopdim > L::MMAX && wide > 16 * 256) {
      L_REG(true);
      MLG_CHECK_HIP(hipGetLastError());
      return 0;
    }
  }
  if (g.ntchopdim > L::MMAX) {
    L_WIDE(true);
  } else if constexpr (L::MMAX > 0) {
    if (wide <= 3 * 256)
      L_WIDE(false);
    else if constexpr (L::N == 256)
      hipLaunchKernelGGL(k_fused_products_256<LINEAR>, dim3(xcd_grid((g.ndimr + 7) / 8 * g.ndimx)), dim3(256), 0,
                         c->stream, g, c->d.r, c->d.tw_t, c->d.tw_h, io, two_omega, n2);
    else
      L_REG(false);
  }
#undef L_WIDE
#undef L_REG
  MLG_CHECK_HIP(hipGetLastError());
  return 0;
}
template <class L>
static int launch_lines(mlg_ctx *c, const FusedIO &io, double two_omega, double n2, int linear) {
  return linear ? launch_line<L, true>(c, io, two_omega, n2) : launch_line<L, false>(c, io, two_omega, n2);
}

int launch_fused_products(mlg_ctx *c, const double2 *const in[10], double2 *const out[4], double two_omega, double n2,
                          int linear, double *zl) {
  KGrid g = kgrid(c);
  FusedIO io;
  for (int i = 0; i < 10; i++) io.in[i] = in[i];
  for (int i = 0; i < 4; i++) io.out[i] = out[i];
  io.zl = zl;
  // PFP traffic: 9 (10) live input fields read, 4 written
  KScope ks(c, K_PRODUCTS, 16.0 * g.nr * g.ntchopdim * (double)g.nx * ((linear ? 10 : 9) + 4));
  switch (g.nth) {
    case 2: return launch_lines<LineTiny<2>>(c, io, two_omega, n2, linear);
    case 4: return launch_lines<LineTiny<4>>(c, io, two_omega, n2, linear);
    case 8: return launch_lines<LineTiny<8>>(c, io, two_omega, n2, linear);
    case 16: return launch_lines<Line16>(c, io, two_omega, n2, linear);
    case 32: return launch_lines<Line32>(c, io, two_omega, n2, linear);
    case 64: return launch_lines<Line64>(c, io, two_omega, n2, linear);
    case 128: return launch_lines<Line128>(c, io, two_omega, n2, linear);
    case 256: return launch_lines<Line256>(c, io, two_omega, n2, linear);
    case 512: return launch_lines<Line512>(c, io, two_omega, n2, linear);
    default: break;
  }
  if (c->fp.n) return launch_fused_any(c, io, two_omega, n2, linear);
  return MLG_E_ARG;
}

}  // namespace mlg
