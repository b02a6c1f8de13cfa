// The poles of the rational approximation of x^-1/2 (funcm.hip): computed on the
// host, read by the kernels from a table in the context's own device memory.
#pragma once
#include <math.h>

#include <vector>

namespace oakg {

constexpr int kPoles = 31;    // pole 31 of a set is s = 0 (T itself)
constexpr int kBuckets = 25;  // kappa = 4, 16, ... 4^25
constexpr int kPoleSet = 64;  // doubles of a set: the poles, then the weights

// Poles and weights for [1, kappa], in extended precision.  With k =
// kappa^-1/2 the zeros and poles are -c_j, c_j = sc^2(j K' / 62) (modulus
// k' = sqrt(1 - k^2)), by the descending Landen transformation for the lower
// half and c_{62-j} = kappa / c_j for the upper one.
inline void zolotarev(long double kappa, double* s, double* w) {
  constexpr int K = kPoles;
  const long double k = 1.0L / sqrtl(kappa);
  long double a[24], c[24];
  int n = 0;
  a[0] = 1.0L;
  c[0] = sqrtl(1.0L - k * k);
  long double b = k;
  while (n < 22 && fabsl(c[n]) > 1e-20L * a[n]) {
    a[n + 1] = (a[n] + b) / 2;
    c[n + 1] = (a[n] - b) / 2;
    b = sqrtl(a[n] * b);
    ++n;
  }
  const long double Kp = 2.0L * atanl(1.0L) / a[n];  // (pi / 2) / AGM(1, k)
  long double cj[2 * K];
  for (int j = 1; j <= K; ++j) {
    long double phi = ldexpl(a[n] * (j * Kp / (2 * K)), n);
    for (int i = n; i >= 1; --i) phi = (phi + asinl(c[i] * sinl(phi) / a[i])) / 2;
    const long double t = tanl(phi);
    cj[j] = t * t;
  }
  cj[K] = sqrtl(kappa);
  for (int j = K + 1; j < 2 * K; ++j) cj[j] = kappa / cj[2 * K - j];
  long double wl[K];
  for (int l = 0; l < K; ++l) {
    long double v = 1.0L;
    for (int i = 0; i < K; ++i) {
      if (i < K - 1) v *= cj[2 * i + 2] - cj[2 * l + 1];
      if (i != l) v /= cj[2 * i + 1] - cj[2 * l + 1];
    }
    wl[l] = v;
  }
  // the relative error equioscillates: scale to its midpoint
  long double lo = 1e30L, hi = 0.0L;
  for (int g = 0; g <= 2000; ++g) {
    const long double x = powl(kappa, g / 2000.0L);
    long double f = 0.0L;
    for (int l = 0; l < K; ++l) f += wl[l] / (x + cj[2 * l + 1]);
    f *= sqrtl(x);
    lo = fminl(lo, f);
    hi = fmaxl(hi, f);
  }
  for (int l = 0; l < K; ++l) {
    s[l] = (double)cj[2 * l + 1];
    w[l] = (double)(wl[l] * 2.0L / (lo + hi));
  }
  s[K] = 0.0;
  w[K] = 0.0;
}

// The table: the sets of all buckets one after another.  The same for every
// device and context, so computed once per process (its host copy never changes).
inline const std::vector<double>& pole_table() {
  static const std::vector<double> table = [] {
    std::vector<double> t((size_t)kBuckets * kPoleSet);
    long double kappa = 1.0L;
    for (int b = 0; b < kBuckets; ++b) {
      kappa *= 4.0L;
      zolotarev(kappa, &t[(size_t)b * kPoleSet], &t[(size_t)b * kPoleSet + 32]);
    }
    return t;
  }();
  return table;
}

}  // namespace oakg
