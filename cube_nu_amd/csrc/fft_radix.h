// fft_radix.h -- register-resident R-point DFTs for the size-specialised FFT
// passes (fft_plane.h, fft_line.hip: R = 2..18; fft_box.hip: 24 and 32).
//
// R = 2, 3, 4, 5, 8 and 16 have their own butterflies; 7, 11 and 13 pair the
// inputs m and R-m (half the products of the plain DFT); the other R = A B are
// B-point DFTs over stride A, constant twiddles and A-point DFTs.  All
// constants are compile-time values.  Complex products are two multiplies and
// two fused multiply-adds.
#pragma once
#include "common.h"

namespace cube {
namespace fftr {

template <typename C>
struct CT;
template <>
struct CT<float2> {
  using R = float;
  __device__ static float2 mk(float a, float b) { return make_float2(a, b); }
};
template <>
struct CT<double2> {
  using R = double;
  __device__ static double2 mk(double a, double b) { return make_double2(a, b); }
};
__device__ inline float fm(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ inline double fm(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename C>
__device__ inline C add(C a, C b) { return CT<C>::mk(a.x + b.x, a.y + b.y); }
template <typename C>
__device__ inline C sub(C a, C b) { return CT<C>::mk(a.x - b.x, a.y - b.y); }
template <typename C>
__device__ inline C mul(C a, C b) { return CT<C>::mk(fm(a.x, b.x, -(a.y * b.y)), fm(a.x, b.y, a.y * b.x)); }
template <typename C>
__device__ inline C scl(C a, typename CT<C>::R s) { return CT<C>::mk(a.x * s, a.y * s); }
template <typename C>
__device__ inline C axpy(typename CT<C>::R s, C a, C b) { return CT<C>::mk(fm(s, a.x, b.x), fm(s, a.y, b.y)); }  // s a + b
template <typename C>
__device__ inline C cj(C a) { return CT<C>::mk(a.x, -a.y); }
// i SIGN a
template <int SIGN, typename C>
__device__ inline C mi(C a) { return SIGN > 0 ? CT<C>::mk(-a.y, a.x) : CT<C>::mk(a.y, -a.x); }
// a W with W the forward twiddle e^{-i t}, conjugated for the inverse
template <int SIGN, typename C>
__device__ inline C mulw(C a, C w) { return mul(a, SIGN > 0 ? cj(w) : w); }

// a / d from inv = 1 / d: the product and one correction by the remainder, the
// rounding of the division (3 operations instead of the 10 of an exact one).
__device__ inline float div_by(float a, float d, float inv) {
  const float q = a * inv;
  return __builtin_fmaf(__builtin_fmaf(-q, d, a), inv, q);
}
__device__ inline double div_by(double a, double d, double) { return a / d; }

// e^{2 pi i k/n} as compile-time values: the angle reduced to [0, pi/4] by
// the octant symmetries, then the Taylor series.
struct CS {
  double c, s;
};
constexpr CS unit(long k, long n) {
  k %= n;
  if (2 * k > n) {
    const CS u = unit(n - k, n);
    return {u.c, -u.s};
  }
  if (4 * k > n) {
    const CS u = unit(n - 2 * k, 2 * n);
    return {-u.c, u.s};
  }
  if (8 * k > n) {
    const CS u = unit(n - 4 * k, 4 * n);
    return {u.s, u.c};
  }
  const double x = 2.0 * kPi * (double)k / (double)n;
  double c = 0, s = 0, t = 1;
  for (int i = 0; i < 24; i += 2) {
    c += (i % 4 == 0) ? t : -t;
    t *= x / (i + 1);
    s += (i % 4 == 0) ? t : -t;
    t *= x / (i + 2);
  }
  return {c, s};
}
template <int R>
struct Roots {
  double c[R], s[R];
};
template <int R>
constexpr Roots<R> roots() {
  Roots<R> t{};
  for (int k = 0; k < R; ++k) {
    const CS u = unit(k, R);
    t.c[k] = u.c;
    t.s[k] = u.s;
  }
  return t;
}

// cos(2 pi k/R) of an odd prime R in FP32 such that k = 1..(R-1)/2 add up to -1/2 exactly,
// as the cosines do: what their roundings leave over (13: 6.7e-8) turns into waves of a
// constant line, and the longest of them outweigh all other errors of a potential
// (coarse kicks of 312^3, 78 points, 2.3 times as far off as by the generic passes).  One
// ulp at a time goes where it adds least to the squares of the errors.
template <int R>
struct Cosines {
  float c[R];
};
constexpr double ulp_below_one(double a) {
  double u = 1.0 / (1 << 24);
  for (a = a < 0 ? -a : a; a < 0.5; a *= 2) u /= 2;
  return u;
}
template <int R>
constexpr Cosines<R> balanced_cosines() {
  constexpr Roots<R> W = roots<R>();
  constexpr int M = (R - 1) / 2;
  double c[M + 1] = {}, left = -0.5;
  for (int k = 1; k <= M; ++k) {
    c[k] = (double)(float)W.c[k];
    left -= c[k];
  }
  while (left != 0) {
    int best = 0;
    double cost = 0, step = 0;
    for (int k = 1; k <= M; ++k) {
      const double u = ulp_below_one(c[k]), d = left > 0 ? u : -u, e = c[k] - W.c[k], q = (e + d) * (e + d) - e * e;
      if (u <= (left > 0 ? left : -left) && (best == 0 || q < cost)) {
        best = k;
        cost = q;
        step = d;
      }
    }
    c[best] += step;
    left -= step;
  }
  Cosines<R> t{};
  t.c[0] = 1.0f;
  for (int k = 1; k <= M; ++k) t.c[k] = t.c[R - k] = (float)c[k];
  return t;
}

template <int SIGN, int R, typename C>
__device__ inline void bfly(C* v);

// 4-point DFT of (a, b, c, d) in place
template <int SIGN, typename C>
__device__ inline void dft4(C& a, C& b, C& c, C& d) {
  const C p = add(a, c), q = sub(a, c), r = add(b, d), t = mi<SIGN>(sub(b, d));
  a = add(p, r);
  c = sub(p, r);
  b = add(q, t);
  d = sub(q, t);
}

// R = A B: X[k1 + B k2] = sum_r W_A^{r k2} W_R^{r k1} sum_m W_B^{m k1} v[r + A m]
template <int SIGN, int A, int B, typename C>
__device__ inline void bfly_ab(C* v) {
  using RR = typename CT<C>::R;
  constexpr int R = A * B;
  constexpr Roots<R> W = roots<R>();
  C u[R];
#pragma unroll
  for (int r = 0; r < A; ++r) {
    C t[B];
#pragma unroll
    for (int m = 0; m < B; ++m) t[m] = v[r + A * m];
    bfly<SIGN, B>(t);
#pragma unroll
    for (int k = 0; k < B; ++k) u[r * B + k] = t[k];
  }
#pragma unroll
  for (int k1 = 0; k1 < B; ++k1) {
    C t[A];
#pragma unroll
    for (int r = 0; r < A; ++r) {
      const int e = r * k1;  // < R
      const C a = u[r * B + k1];
      t[r] = e == 0 ? a
                    : (4 * e == R ? mi<SIGN>(a)
                                  : mul(a, CT<C>::mk((RR)W.c[e], SIGN > 0 ? (RR)W.s[e] : (RR)(-W.s[e]))));
    }
    bfly<SIGN, A>(t);
#pragma unroll
    for (int k2 = 0; k2 < A; ++k2) v[k1 + B * k2] = t[k2];
  }
}

// odd prime R: X_k = v_0 + sum_m cos(2 pi m k/R) (v_m + v_{R-m}) +- i sum_m sin(..) (v_m - v_{R-m})
template <int SIGN, int R, typename C>
__device__ inline void bfly_prime(C* v) {
  using RR = typename CT<C>::R;
  constexpr Roots<R> W = roots<R>();
  constexpr Cosines<R> W32 = balanced_cosines<R>();
  constexpr int M = (R - 1) / 2;
  auto cosine = [&](int e) -> RR { return sizeof(RR) == 4 ? (RR)W32.c[e] : (RR)W.c[e]; };
  C a[M], b[M], s0 = v[0];
#pragma unroll
  for (int m = 0; m < M; ++m) {
    a[m] = add(v[m + 1], v[R - 1 - m]);
    b[m] = sub(v[m + 1], v[R - 1 - m]);
    s0 = add(s0, a[m]);
  }
#pragma unroll
  for (int k = 1; k <= M; ++k) {
    C p = v[0], q = CT<C>::mk((RR)0, (RR)0);
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int e = ((m + 1) * k) % R;
      p = axpy(cosine(e), a[m], p);
      q = m == 0 ? scl(b[m], (RR)W.s[e]) : axpy((RR)W.s[e], b[m], q);
    }
    q = mi<SIGN>(q);
    // v[k], v[R-k] were read into a, b; v[0] is still the input
    v[k] = add(p, q);
    v[R - k] = sub(p, q);
  }
  v[0] = s0;
}

template <int SIGN, int R, typename C>
__device__ inline void bfly(C* v) {
  using RR = typename CT<C>::R;
  if constexpr (R == 1) {
  } else if constexpr (R == 2) {
    const C a = v[0], b = v[1];
    v[0] = add(a, b);
    v[1] = sub(a, b);
  } else if constexpr (R == 4) {
    dft4<SIGN>(v[0], v[1], v[2], v[3]);
  } else if constexpr (R == 3) {
    const C t = add(v[1], v[2]);
    const C m = axpy((RR)-0.5, t, v[0]);
    const C r = mi<SIGN>(scl(sub(v[1], v[2]), (RR)0.86602540378443864676));
    v[0] = add(v[0], t);
    v[1] = add(m, r);
    v[2] = sub(m, r);
  } else if constexpr (R == 5 || R == 7 || R == 11 || R == 13) {
    bfly_prime<SIGN, R>(v);
  } else if constexpr (R == 8) {
    C e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4<SIGN>(e0, e1, e2, e3);
    dft4<SIGN>(o0, o1, o2, o3);
    const RR h = (RR)0.70710678118654752440;
    // W8 o1 = h (o1 +- i o1), W8^3 o3 = h (-o3 +- i o3)
    o1 = scl(add(o1, mi<SIGN>(o1)), h);
    o2 = mi<SIGN>(o2);
    o3 = scl(sub(mi<SIGN>(o3), o3), h);
    v[0] = add(e0, o0);
    v[4] = sub(e0, o0);
    v[1] = add(e1, o1);
    v[5] = sub(e1, o1);
    v[2] = add(e2, o2);
    v[6] = sub(e2, o2);
    v[3] = add(e3, o3);
    v[7] = sub(e3, o3);
  } else if constexpr (R == 16) {
    bfly_ab<SIGN, 4, 4>(v);
  } else if constexpr (R % 4 == 0) {
    bfly_ab<SIGN, R / 4, 4>(v);  // 12
  } else if constexpr (R % 3 == 0) {
    bfly_ab<SIGN, R / 3, 3>(v);  // 6, 9, 15, 18
  } else {
    static_assert(R % 2 == 0, "radix");
    bfly_ab<SIGN, R / 2, 2>(v);  // 10, 14
  }
}

// N = r1 r2 with both factors <= kMaxRadix, as near to square as possible;
// r1 takes the odd factor where there is one (a stage writes with stride r1).
constexpr int kMaxRadix = 18;
constexpr bool radix_ok(int r) {
  return r == 1 || r == 2 || r == 3 || r == 4 || r == 5 || r == 6 || r == 7 || r == 8 || r == 9 || r == 10 ||
         r == 11 || r == 12 || r == 13 || r == 14 || r == 15 || r == 16 || r == 18;
}
struct Split {
  int r1, r2;
};
constexpr Split split2(int n) {
  Split best{0, 0};
  int cost = 1 << 30;
  for (int a = 1; a <= kMaxRadix; ++a) {
    if (n % a != 0 || !radix_ok(a) || n / a > kMaxRadix || !radix_ok(n / a)) continue;
    const int b = n / a;
    const int c = 4 * (a > b ? a : b) + (a % 2 ? 0 : 1);
    if (c < cost) {
      cost = c;
      best = Split{a, b};
    }
  }
  return best;
}

}  // namespace fftr
}  // namespace cube
