// Register butterflies of the mixed-radix FFT kernels (device code only).
#pragma once
#include <hip/hip_runtime.h>

namespace mlg {
namespace fftr {

#pragma clang fp contract(fast)

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
// a times the root w, or its conjugate for the inverse transform
template <bool INV>
__device__ __forceinline__ double2 rmul(double2 a, double2 w) {
  return INV ? make_double2(a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y) : cmul(a, w);
}
__device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
// -i a (forward) or i a (inverse)
template <bool INV>
__device__ __forceinline__ double2 mulj(double2 a) {
  return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// e^{-2 pi i k / R} for the small radices, whose roots are written out
template <int R>
__device__ __forceinline__ constexpr double root_x(int k) {
  constexpr double c3[3] = {1.0, -0.5, -0.5};
  constexpr double c5[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410, -0.80901699437494742410,
                            0.30901699437494742410};
  constexpr double c7[7] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624,
                            -0.90096886790241912624, -0.22252093395631440429, 0.62348980185873353053};
  return R == 3 ? c3[k % 3] : R == 5 ? c5[k % 5] : c7[k % 7];
}
template <int R>
__device__ __forceinline__ constexpr double root_y(int k) {
  constexpr double s3[3] = {0.0, -0.86602540378443864676, 0.86602540378443864676};
  constexpr double s5[5] = {0.0, -0.95105651629515357212, -0.58778525229247312917, 0.58778525229247312917,
                            0.95105651629515357212};
  constexpr double s7[7] = {0.0, -0.78183148246802980871, -0.97492791218182360702, -0.43388373911755812048,
                            0.43388373911755812048, 0.97492791218182360702, 0.78183148246802980871};
  return R == 3 ? s3[k % 3] : R == 5 ? s5[k % 5] : s7[k % 7];
}

// R-point DFT, natural order in and out; w[k st] = e^{-2 pi i k / R}
// (uniform over the block: scalar loads; radices up to 8 do not read it).
template <int R, bool INV>
struct Dft;
template <bool INV>
struct Dft<2, INV> {
  static __device__ __forceinline__ void run(double2 (&v)[2], const double2 *, int) {
    const double2 a = v[0];
    v[0] = cadd(a, v[1]);
    v[1] = csub(a, v[1]);
  }
};
template <bool INV>
struct Dft<4, INV> {
  static __device__ __forceinline__ void run(double2 (&v)[4], const double2 *, int) {
    const double2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]), c = cadd(v[1], v[3]), d = mulj<INV>(csub(v[1], v[3]));
    v[0] = cadd(a, c);
    v[1] = cadd(b, d);
    v[2] = csub(a, c);
    v[3] = csub(b, d);
  }
};
// odd prime: outputs k and R - k from the sums and differences of inputs q
// and R - q
template <int R, bool INV>
struct DftPrime {
  static __device__ __forceinline__ void run(double2 (&v)[R], const double2 *__restrict__ w, int st) {
    constexpr int H = (R - 1) / 2;
    double2 a[H], d[H];
    double2 s0 = v[0];
#pragma unroll
    for (int q = 1; q <= H; q++) {
      a[q - 1] = cadd(v[q], v[R - q]);
      d[q - 1] = csub(v[q], v[R - q]);
      s0 = cadd(s0, a[q - 1]);
    }
    double2 c[H];
#pragma unroll
    for (int q = 1; q <= H; q++) {
      if constexpr (R <= 7) c[q - 1] = make_double2(root_x<R>(q), root_y<R>(q));
      else c[q - 1] = w[q * st];
    }
#pragma unroll
    for (int k = 1; k <= H; k++) {
      double2 A = v[0], B = make_double2(0.0, 0.0);
#pragma unroll
      for (int q = 1; q <= H; q++) {
        const int e = (q * k) % R, h = e <= H ? e : R - e;
        const double cx = c[h - 1].x, cy = e <= H ? c[h - 1].y : -c[h - 1].y;
        A.x += a[q - 1].x * cx;
        A.y += a[q - 1].y * cx;
        B.x += d[q - 1].x * cy;
        B.y += d[q - 1].y * cy;
      }
      // forward: A + i B, inverse: A - i B (cy = -sin)
      const double2 jb = INV ? make_double2(B.y, -B.x) : make_double2(-B.y, B.x);
      v[k] = cadd(A, jb);
      v[R - k] = csub(A, jb);
    }
    v[0] = s0;
  }
};
template <bool INV> struct Dft<3, INV> : DftPrime<3, INV> {};
template <bool INV> struct Dft<5, INV> : DftPrime<5, INV> {};
template <bool INV> struct Dft<7, INV> : DftPrime<7, INV> {};
template <bool INV> struct Dft<11, INV> : DftPrime<11, INV> {};
template <bool INV> struct Dft<13, INV> : DftPrime<13, INV> {};
template <bool INV> struct Dft<17, INV> : DftPrime<17, INV> {};
template <bool INV> struct Dft<19, INV> : DftPrime<19, INV> {};
// R = A B: A-point DFTs over stride B, W_R^{j k}, B-point DFTs
template <int A, int B, bool INV>
struct DftProduct {
  static __device__ __forceinline__ void run(double2 (&v)[A * B], const double2 *__restrict__ w, int st) {
    double2 t[B][A];
#pragma unroll
    for (int j = 0; j < B; j++) {
#pragma unroll
      for (int q = 0; q < A; q++) t[j][q] = v[j + B * q];
      Dft<A, INV>::run(t[j], w, st * B);
#pragma unroll
      for (int k = 1; k < A; k++)
        if (j > 0) t[j][k] = rmul<INV>(t[j][k], w[j * k * st]);
    }
#pragma unroll
    for (int k = 0; k < A; k++) {
      double2 u[B];
#pragma unroll
      for (int j = 0; j < B; j++) u[j] = t[j][k];
      Dft<B, INV>::run(u, w, st * A);
#pragma unroll
      for (int j = 0; j < B; j++) v[k + A * j] = u[j];
    }
  }
};
// 6: 3-point DFTs of the even and odd inputs
template <bool INV>
struct Dft<6, INV> {
  static __device__ __forceinline__ void run(double2 (&v)[6], const double2 *, int) {
    constexpr double h = 0.86602540378443864676;
    double2 e[3] = {v[0], v[2], v[4]}, o[3] = {v[1], v[3], v[5]};
    Dft<3, INV>::run(e, nullptr, 0);
    Dft<3, INV>::run(o, nullptr, 0);
    o[1] = rmul<INV>(o[1], make_double2(0.5, -h));
    o[2] = rmul<INV>(o[2], make_double2(-0.5, -h));
#pragma unroll
    for (int k = 0; k < 3; k++) {
      v[k] = cadd(e[k], o[k]);
      v[k + 3] = csub(e[k], o[k]);
    }
  }
};
// 8: 4-point DFTs of the even and odd inputs, roots 1, (1 - i)/sqrt 2, -i, -(1 + i)/sqrt 2
template <bool INV>
struct Dft<8, INV> {
  static __device__ __forceinline__ void run(double2 (&v)[8], const double2 *, int) {
    constexpr double h = 0.70710678118654752440;
    double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    Dft<4, INV>::run(e, nullptr, 0);
    Dft<4, INV>::run(o, nullptr, 0);
    const double2 j1 = mulj<INV>(o[1]), j3 = mulj<INV>(o[3]);
    o[1] = make_double2(h * (o[1].x + j1.x), h * (o[1].y + j1.y));
    o[2] = mulj<INV>(o[2]);
    o[3] = make_double2(h * (j3.x - o[3].x), h * (j3.y - o[3].y));
#pragma unroll
    for (int k = 0; k < 4; k++) {
      v[k] = cadd(e[k], o[k]);
      v[k + 4] = csub(e[k], o[k]);
    }
  }
};
template <bool INV> struct Dft<9, INV> : DftProduct<3, 3, INV> {};
template <bool INV> struct Dft<10, INV> : DftProduct<2, 5, INV> {};
template <bool INV> struct Dft<12, INV> : DftProduct<3, 4, INV> {};
template <bool INV> struct Dft<16, INV> : DftProduct<4, 4, INV> {};

}  // namespace fftr
}  // namespace mlg
