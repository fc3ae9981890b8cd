// Compile-time unit roots of the register DFTs, correctly rounded: sine and
// cosine from their Taylor series after exact octant reduction, evaluated by the
// compiler in pairs of doubles.
#pragma once

namespace qepw {

// Sums and products of two doubles as a double and its rounding error (Dekker).
// In plain doubles the reduced angle and the series were off by up to three
// roundings, the same in every line, so that the errors added up over the passes:
// h_psi in FP64 against 80-bit transforms, 36^3 7.6e-16 with those and 5.9e-16 with
// these, 96^3 1.0e-15 and 5.4e-16, 40 x 36 x 128 5.2e-16 and 3.4e-16 (radix passes
// with exactly rounded twiddles: 3.2e-16).
struct CxPair {
  double h, l;
};
constexpr CxPair cx_add(CxPair a, CxPair b) {
  const double s = a.h + b.h, t = s - a.h;
  const double e = (a.h - (s - t)) + (b.h - t) + a.l + b.l;
  const double h = s + e;
  return {h, e - (h - s)};
}
constexpr CxPair cx_mul(CxPair a, CxPair b) {
  const double split = 134217729.0;  // 2^27 + 1
  const double ta = split * a.h, tb = split * b.h;
  const double ah = ta - (ta - a.h), al = a.h - ah, bh = tb - (tb - b.h), bl = b.h - bh;
  const double p = a.h * b.h;
  const double e =
      ((ah * bh - p) + ah * bl + al * bh) + al * bl + (a.h * b.l + a.l * b.h);
  const double h = p + e;
  return {h, e - (h - p)};
}
constexpr CxPair cx_div(CxPair a, double b) {
  const double q = a.h / b;
  const CxPair r = cx_add(a, cx_mul({-q, 0.0}, {b, 0.0}));
  return cx_add({q, 0.0}, {(r.h + r.l) / b, 0.0});
}
// pi / 4 and its remainder
constexpr CxPair kPi4 = {0.78539816339744830961566084581987572, 3.0616169978683829431e-17};

// sum over i of (-1)^i x^(2 i + odd) / (2 i + odd)!, |x| <= pi/4
constexpr double cx_series(CxPair x, int odd) {
  CxPair term = odd ? x : CxPair{1.0, 0.0}, sum = term;
  const CxPair x2 = cx_mul(x, x);
  for (int i = 1; i < 16; ++i) {
    const double n = 2.0 * i + odd;
    term = cx_div(cx_mul(term, {-x2.h, -x2.l}), n * (n - 1.0));
    sum = cx_add(sum, term);
  }
  return sum.h + sum.l;
}
constexpr double cx_sin_small(CxPair x) { return cx_series(x, 1); }
constexpr double cx_cos_small(CxPair x) { return cx_series(x, 0); }

// cos / sin of 2 pi k / n, k reduced exactly into an octant: theta = (pi/4) (8k/n),
// r = (pi/4) j/n past octant o, q = pi/4 - r.
constexpr CxPair cx_octant(int j, int n) {
  return cx_div(cx_mul(kPi4, {(double)j, 0.0}), (double)n);
}
constexpr double cx_cos2pi(int k, int n) {
  k %= n;
  if (k < 0) k += n;
  const int o = (8 * k) / n, j = 8 * k - o * n;
  const CxPair r = cx_octant(j, n), q = cx_octant(n - j, n);
  switch (o) {
    case 0: return cx_cos_small(r);
    case 1: return cx_sin_small(q);
    case 2: return -cx_sin_small(r);
    case 3: return -cx_cos_small(q);
    case 4: return -cx_cos_small(r);
    case 5: return -cx_sin_small(q);
    case 6: return cx_sin_small(r);
    default: return cx_cos_small(q);
  }
}
constexpr double cx_sin2pi(int k, int n) {
  k %= n;
  if (k < 0) k += n;
  const int o = (8 * k) / n, j = 8 * k - o * n;
  const CxPair r = cx_octant(j, n), q = cx_octant(n - j, n);
  switch (o) {
    case 0: return cx_sin_small(r);
    case 1: return cx_cos_small(q);
    case 2: return cx_cos_small(r);
    case 3: return cx_sin_small(q);
    case 4: return -cx_sin_small(r);
    case 5: return -cx_cos_small(q);
    case 6: return -cx_cos_small(r);
    default: return -cx_sin_small(q);
  }
}

template <int M> struct UnitRoots {
  // w[k] = exp(+2 pi i k / M)
  double c[M > 0 ? M : 1];
  double s[M > 0 ? M : 1];
  constexpr UnitRoots() : c(), s() {
    for (int k = 0; k < M; ++k) {
      c[k] = cx_cos2pi(k, M);
      s[k] = cx_sin2pi(k, M);
    }
  }
};

}  // namespace qepw
