// DIAGNOST's every-IT1 section (src/mod_march.f90:1797-1961) and CALCXY
// (:1967-2047): the domain integrals of vorticity, axial momentum, energy,
// helicity and angular momentum, the spread of psi and chi at r = infinity
// (CALCAT1), and the enstrophy-weighted vortex centre and radius.
//
// The fields are formed by the library's operators at NRCHOP+3; the
// integrals are the first FFF coefficient (INTEG, src/mod_scalar3.f90:
// 312-353), Gauss sums over PFF columns (PRODCT :398-468, the per-(m, k)
// product launch of the energy diagnostics) or sums over the physical grid
// (CALCXY's, of ABSVEC2 :2050-2099 times MULRCOSTH / MULRSINTH / MULR2's
// factors :2102-2225).
#include <algorithm>
#include <cmath>
#include <vector>

#include "mlegs_internal.h"

using namespace mlg;

#define RET(x)                 \
  do {                         \
    int _r = (x);              \
    if (_r) return _r;         \
  } while (0)

namespace mlg {

// ABSVEC2, ((u^2 + v^2) / r^2 + w^2) / (1-x)^2, summed over z per (r, theta):
// out[j][r], the real and the imaginary theta sub-grid.  Block: 64 radial nodes x 4 ranges of z at one theta.
__global__ void __launch_bounds__(256) k_absvec2_sum(KGrid g, const double2 *__restrict__ u, const double2 *__restrict__ v,
                                                     const double2 *__restrict__ w, const double *__restrict__ r2,
                                                     const double *__restrict__ x, double2 *__restrict__ out) {
  __shared__ double2 S[4][64];
  const int rl = threadIdx.x & 63, q = threadIdx.x >> 6, r = blockIdx.x * 64 + rl, j = blockIdx.y;
  double2 s = make_double2(0.0, 0.0);
  if (r < g.nr) {
    const double om = 1 - x[r], f = om * om, rr = r2[r];
    for (int z = q; z < g.nx; z += 4) {
      const size_t at = (size_t)r + (size_t)g.ndimr * ((size_t)j + (size_t)g.ndimth * z);
      const double2 uu = u[at], vv = v[at], ww = w[at];
      s.x += ((uu.x * uu.x + vv.x * vv.x) / rr + ww.x * ww.x) / f;
      s.y += ((uu.y * uu.y + vv.y * vv.y) / rr + ww.y * ww.y) / f;
    }
  }
  S[q][rl] = s;
  __syncthreads();
  if (q == 0 && r < g.nr)
    out[(size_t)r + (size_t)g.nr * j] = make_double2(S[0][rl].x + S[1][rl].x + S[2][rl].x + S[3][rl].x,
                                                     S[0][rl].y + S[1][rl].y + S[2][rl].y + S[3][rl].y);
}

// Inputs of k_it1_values; every sum of the section in one launch.
struct It1 {
  const double2 *dp, *dc, *ang;  // FFF: DELSQH(psi) = -OZ/(1-x)^2, DELSQH(chi) = -UZ/(1-x)^2, XXDX(psi)
  const double2 *f[2];             // psi, chi
  const double *at1, *x, *w, *r2, *terms;  // terms: the PRODCTs' per-(m, k) sums, 3 x na
  const double2 *abs;              // ABSVEC2 summed over z, [theta][r]
  double p00;                      // P_0^0, normalised
  int na, nn;                      // nn: NRCHOP
  long nfff;                       // stored coefficients
  double minc;
};
// VALVOR, VALZMO, the INTEG_P sum, 3 PRODCTs, 4 moments (1, x, y, r^2), then
// CALCAT1's |value| per k of psi and of chi, from value q0 on; a block of 1024 threads each
__global__ void __launch_bounds__(1024) k_it1_values(KGrid g, It1 v, double *out, int q0) {
  __shared__ double2 S[1024];
  const int t = threadIdx.x, q = q0 + blockIdx.x;
  double2 s = make_double2(0.0, 0.0);
  if (q < 2) {
    if (t == 0) s.x = -(q == 0 ? v.dp : v.dc)[0].x;
  } else if (q == 2) {
    // the first NR stored coefficients in storage order
    for (int i = t; i < min((long)g.nr, v.nfff); i += 1024) {
      const double om = 1 - v.x[i];
      s.x += v.ang[i].x / (om * om) * v.w[i];
    }
  } else if (q < 6) {
    for (int i = t; i < v.na; i += 1024) s.x += v.terms[(size_t)(q - 3) * v.na + i];
  } else if (q < IT1_FIXED) {
    // The (0, 0, 0) coefficient of ABSVEC2 times the factor: HORFFT's m = 0
    // and VERFFT's k = 0 are means, RTRAN's n = 0 the Gauss sum with P_0^0.
    // theta = 2 pi j / NTH in the real slots, 2 pi (j + 1/2) / NTH in the imaginary ones
    const double pi = 3.14159265358979323846;
    for (long i = t; i < (long)g.nr * g.nth; i += 1024) {
      const int r = (int)(i % g.nr), j = (int)(i / g.nr);
      double2 a = v.abs[i];
      const double rad = q == 6 ? 1.0 : (q == 9 ? v.r2[r] : sqrt(v.r2[r]));
      if (q == 7 || q == 8) {
        const double thr = 2 * pi / v.minc / g.nth * j, thi = 2 * pi / v.minc / g.nth * (j + 0.5);
        a.x *= q == 7 ? cos(thr) : sin(thr);
        a.y *= q == 7 ? cos(thi) : sin(thi);
      }
      s.x += v.w[r] * rad * (a.x + a.y);
    }
  } else {
    const int k = (q - IT1_FIXED) % g.nxchopdim, fi = (q - IT1_FIXED) / g.nxchopdim;
    const double2 *col = v.f[fi] + (size_t)g.nrchopdim * g.ntchopdim * k;
    for (int n = t; n < v.nn; n += 1024) {
      s.x += col[n].x * v.at1[n];
      s.y += col[n].y * v.at1[n];
    }
  }
  S[t] = s;
  __syncthreads();
  for (int h = 512; h > 0; h >>= 1) {
    if (t < h) S[t] = make_double2(S[t].x + S[t + h].x, S[t].y + S[t + h].y);
    __syncthreads();
  }
  if (t) return;
  if (q >= IT1_FIXED) out[q] = hypot(S[0].x, S[0].y);
  else if (q >= 6) out[q] = S[0].x * v.p00 / (2.0 * g.nth * g.nx);
  else out[q] = S[0].x;
}

// The section without a wait or a host table on the way: every integral ends
// in k_it1_values, whose results come in one copy.  CALCXY's four integrals
// are sums of ABSVEC2 over the physical grid with their factors, in place of
// four fields transformed for one coefficient each (MULRCOSTH / MULRSINTH /
// MULR2 and INTEG), and the eight fields that leave FFF share one backward
// launch.  At 128x64x64 the section with the energies and ENEMON, which share
// launches in the same way, takes 0.39 ms where they took 1.86.  The fields
// lie in seven buffers, one routine's at a time where they would not fit.
static int diagnost_it1(const mlg_field *psi, const mlg_field *chi, double *out) {
  mlg_ctx *c = psi->ctx;
  const Grid &G = c->g;
  const double pi = 3.14159265358979323846;
  const long nf = c->n_fff, np = c->n_pff;
  const size_t na = (size_t)G.ntchop * G.nxchopdim;
  // LN: zero, 2 psi's, then those of a, d2c, dc, dp, ror, rop, oz and scratch
  double *const lnv = c->d.lnv, *const l2 = lnv + 1, *const la = lnv + 2, *const ld2 = lnv + 3, *const ldc = lnv + 4,
               *const ldp = lnv + 5, *const lr = lnv + 6, *const lp = lnv + 7, *const lo = lnv + 8, *const lx = lnv + 9;
  Temps T(c);
  Pack P(T, 7, 3);
  // p: PFF of a, psi, d2c, dc, dp and the vorticity; the first three buffers
  // take the vorticity in physical space once what is packed there is done with
  double2 *p[8], *dp, *dc, *ang, *sum, *a, *d2c, *ror, *rop, *oz, *m1, *vor[3];
  for (int q = 0; q < 8; q++) p[q] = P.take(np, q >= 5);
  dp = P.take(nf, true), dc = P.take(nf, true), ang = P.take(nf, true), sum = P.take((long)G.nr * G.nth, true);
  a = P.take(nf), d2c = P.take(nf), ror = P.take(nf), rop = P.take(nf), oz = P.take(nf);
  m1 = p[0];
  PffProducts q{c, !P.ok};
  if (q.lean) {
    P.grow(6);
    dp = p[7] = P.e[0];
    dc = ror = P.e[1];
    ang = a = d2c = rop = P.e[2];
    p[0] = p[2] = m1 = p[5] = sum = P.e[3];
    p[1] = p[3] = oz = P.e[4];
    p[4] = p[6] = P.e[5];
  }
  for (int i = 0; i < 3; i++) vor[i] = q.lean ? (i == 0 ? ror : i == 1 ? rop : oz) : P.e[i];
  RET(T.ready());
  It1 v;
  v.f[0] = psi->e, v.f[1] = chi->e;
  v.at1 = c->d.at1, v.x = c->d.x, v.w = c->d.w, v.r2 = c->d.r, v.terms = c->d.red;
  v.dp = dp, v.dc = dc, v.ang = ang, v.abs = sum;
  v.p00 = G.pf[0];
  v.na = (int)na, v.nn = G.nrchop, v.nfff = nf;
  v.minc = G.p.minc;
  const int nxd = G.nxchopdim, nval = IT1_FIXED + 2 * nxd, nfff = 3;  // the first nfff values read FFF fields
  auto values = [&](int q0, int q1) -> int {
    hipLaunchKernelGGL(k_it1_values, dim3(q1 - q0), dim3(1024), 0, c->stream, kgrid(c), v, c->d.it1, q0);
    MLG_CHECK_HIP(hipGetLastError());
    return 0;
  };
  // PC2VOR(..., 'H')'s OZ/(1-x)^2 = -DELSQH(psi); PC2VEL(..., 'H'): only
  // UZ/(1-x)^2 = -DELSQH(chi) is read (INTEG)
  RET(launch_delsqh(c, psi->e, psi->ln, dp, ldp));
  RET(launch_delsqh(c, chi->e, chi->ln, dc, ldc));
  // VALANG = -INTEG_P(XXDX(psi with LN = 0)).  INTEG_P (src/mod_march.f90:
  // 3649-3682) sums Re(F%E(:NR,1,1)) w / (1-x)^2 of its FFF argument: the
  // first NR stored coefficients in storage order (past the m = 0, k = 0
  // column when NRCHOPDIM < NR), as the reference reads them
  RET(launch_band3(c, 1, psi->e, lnv, ang, lx));
  if (q.lean) RET(values(0, nfff));
  // VALENE = -PRODCT(DELSQH(psi, 2 LN), psi) + PRODCT(DELSQH(chi), DEL2(chi)),
  // VALHEL = 2 PRODCT(DELSQH(psi), DEL2(chi))
  RET(launch_set_ln(c, l2, psi->ln, 2.0, 0.0));
  RET(launch_delsqh(c, psi->e, l2, a, la));
  q.field(a, la, p[0]);
  q.field(psi->e, lnv, p[1]);
  q.term(p[0], p[1], 0, c->d.red);
  RET(q.group());
  RET(launch_check_top_m1(c, chi->e));
  RET(launch_del2(c, chi->e, chi->ln, d2c, ld2));
  q.field(d2c, ld2, p[2]);
  q.field(dc, ldc, p[3]);
  q.field(dp, ldp, p[4]);
  q.term(p[3], p[2], 0, c->d.red + na);
  q.term(p[4], p[2], 0, c->d.red + 2 * na);
  RET(q.group());
  // the vorticity: ROR, ROP of PC2VOR; OZH (1-x)^2 = OZ, but for its sign,
  // which ABSVEC2 squares
  RET(launch_pc2vor(c, psi->e, psi->ln, chi->e, chi->ln, ror, rop, oz, lr, lp, lx));
  RET(launch_band3(c, 0, dp, ldp, m1, lx));
  RET(launch_band3(c, 0, m1, lx, oz, lo));
  q.field(ror, lr, p[5]);
  q.field(rop, lp, p[6]);
  q.field(oz, lo, p[7]);
  RET(q.flush());
  // CALCXY: the vorticity to physical space
  const double2 *vin[3] = {p[5], p[6], p[7]};
  RET(launch_verfft_bwd_n(c, 3, vin, vor));
  RET(launch_horfft_bwd_n(c, 3, vor, 1.0, 1.0, nullptr));
  hipLaunchKernelGGL(k_absvec2_sum, dim3((G.nr + 63) / 64, G.nth), dim3(256), 0, c->stream, kgrid(c), vor[0], vor[1], vor[2],
                     c->d.r, c->d.x, sum);
  MLG_CHECK_HIP(hipGetLastError());
  RET(values(q.lean ? nfff : 0, nval));
  std::vector<double> h(nval);
  MLG_CHECK_HIP(hipMemcpyAsync(h.data(), c->d.it1, sizeof(double) * nval, hipMemcpyDeviceToHost, c->stream));
  MLG_CHECK_HIP(hipStreamSynchronize(c->stream));
  // INTEG (src/mod_scalar3.f90:312-353): 4 pi ZLEN ELL^2 Re(f(0,0,0)) NORM(0, m=0)
  const double fi = 4.0 * pi * G.zlen * G.ell2;
  out[0] = fi * h[0] * G.norm[0];  // VALVOR
  out[1] = fi * h[1] * G.norm[0];  // VALZMO
  out[2] = -h[3] + h[4];           // VALENE
  out[3] = 2 * h[5];               // VALHEL
  out[4] = -(2.0 * pi * G.zlen * G.ell2 * h[2]);
  // psi and chi at r = infinity (CALCAT1, src/mod_scalar3.f90:286-310)
  for (int q = 0; q < 2; q++) {
    const double *at = h.data() + IT1_FIXED + q * nxd;
    out[5 + 2 * q] = at[0];
    out[6 + 2 * q] = *std::max_element(at, at + nxd) - *std::min_element(at, at + nxd);
  }
  out[9] = h[7] / h[6];              // <X>
  out[10] = h[8] / h[6];             // <Y>
  out[11] = std::sqrt(h[9] / h[6]);  // <R>
  return 0;
}

}  // namespace mlg

// out: VALVOR, VALZMO, VALENE, VALHEL, VALANG, |PSIAT1(k=0)|, spread of
// |PSIAT1|, |CHIAT1(k=0)|, spread of |CHIAT1|, <X>, <Y>, <R>
extern "C" int mlg_diagnost_it1(const mlg_field *psi, const mlg_field *chi, double out[12]) {
  if (!psi || !chi || !out || chi->ctx != psi->ctx) return MLG_E_ARG;
  if (psi->space != MLG_FFF || chi->space != MLG_FFF) return MLG_E_SPACE;
  mlg_ctx *c = psi->ctx;
  RET(mlg_chopset(c, 3));
  const int rc = diagnost_it1(psi, chi, out);
  mlg_chopset(c, -3);
  RET(rc);
  return mlg_synchronize(c);
}
