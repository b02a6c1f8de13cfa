// The poles of the rational approximation of x^-1/2 (funcm.hip): computed on the
// host, read by the kernels from a table in the context's own device memory.
//
// x^-1/2 on [1, kappa] = sum_j w_j / (x + s_j), j = 0 .. K-1: with k = kappa^-1/2,
// k'^2 = 1 - k^2, y_j = (j + 1/2) K(k') / K and elliptic functions of modulus k',
//
//   s_j = sc^2(y_j),  w_j = 2 K(k') / (pi K) dn(y_j) nc^2(y_j)
//
// (Hale, Higham and Trefethen, SIAM J. Numer. Anal. 46, 2008, method 3; these are
// Zolotarev's poles).  Relative error 4 exp(-2 pi^2 K / log(16 kappa)):
//
//   31 poles   kappa = 4^9 1.5e-17, 4^10 4.2e-16, 4^11 7e-15, 4^15 3e-10, 4^25 3e-7
//   63 poles   kappa = 4^20 8e-18, 4^22 2.3e-16
//
// The table: blocks of 32 poles and their weights, for kappa = 4, 16, ... one block
// each up to 4^10 (pole 31 is s = 0, T itself, with weight 0), two each up to 4^22,
// of which the first ends with s = 0 as well.  (The spectrum's own power of 4, not
// one interval for all: in x^1/2 c = sum_j w_j (c - s_j (x + s_j)^-1 c) the poles far
// above the spectrum cost (s_j / x)^1/2 in rounding.)  At 4^22 rounding M has moved
// its small eigenvalues by eps kappa = 4e-3; beyond, they need not be positive any
// more, and no sum of shifted solves stands for a function of eigenvalues that
// are cut off at 1: the eigenvalues themselves are taken.
#pragma once
#include <math.h>

#include <vector>

#ifdef __HIPCC__
#define OAK_HD __host__ __device__
#else
#define OAK_HD
#endif

namespace oakg {

constexpr int kPoleBlock = 64;  // doubles of a block: 32 poles, 32 weights
constexpr int kOneBlock = 10, kTwoBlocks = 22;  // kappa up to 4^kOneBlock: one block, ...

// The blocks for a spectrum in [1, 2^ex): first .. first + count - 1; count 0: none.
struct PoleBlocks {
  int first, count;
};
OAK_HD inline PoleBlocks pole_blocks(int ex) {
  const int b = ex < 3 ? 1 : (ex + 1) >> 1;  // 4^b >= 2^ex
  if (b <= kOneBlock) return PoleBlocks{b - 1, 1};
  if (b <= kTwoBlocks) return PoleBlocks{2 * b - kOneBlock - 2, 2};
  return PoleBlocks{0, 0};
}

// cs and dn of modulus k' as sums over the poles of their period (K: K(k), the
// imaginary quarter period; all terms of dn are positive, and those of cs fall
// from the first on by more than e^2), for y <= K(k') / 2, the other half
// by the quarter-period shift: sc(K(k') - y) = cs(y) / k, dn(K(k') - y) = k / dn(y).
inline void inv_sqrt_poles(long double kappa, int K, double* s, double* w) {
  const long double pi = 3.14159265358979323846264338327950288L;
  const long double k = 1.0L / sqrtl(kappa);
  auto quarter = [pi](long double b) {  // (pi / 2) / AGM(1, b)
    long double a = 1.0L;
    for (int i = 0; i < 40; ++i) {
      const long double t = (a + b) / 2;
      b = sqrtl(a * b);
      a = t;
    }
    return pi / (2 * a);
  };
  const long double c = pi / (2 * quarter(sqrtl(1.0L - k * k))), Kp = quarter(k);
  for (int j = 0; j < K; ++j) {
    const long double y = (j + 0.5L) * Kp / K, yl = fminl(y, Kp - y);
    long double cs = 0.0L, dn = 0.0L;
    for (int n = -20; n <= 20; ++n) {
      const long double a = c * (yl - 2 * n * Kp);
      if (fabsl(a) > 60.0L) continue;
      cs += c / sinhl(a);
      dn += c / coshl(a);
    }
    const bool low = y == yl;
    const long double sj = low ? 1.0L / (cs * cs) : kappa * cs * cs;
    s[j] = (double)sj;
    w[j] = (double)(2 * Kp / (pi * K) * (low ? dn : k / dn) * (1.0L + sj));
  }
}

// The same for every device and context, so computed once per process (2 ms; the
// host copy never changes).
inline const std::vector<double>& pole_table() {
  static const std::vector<double> table = [] {
    std::vector<double> t((size_t)(2 * kTwoBlocks - kOneBlock) * kPoleBlock, 0.0);
    long double kappa = 1.0L;
    for (int b = 1; b <= kTwoBlocks; ++b) {
      kappa *= 4.0L;
      const PoleBlocks pb = pole_blocks(2 * b);
      const int K = 32 * pb.count - 1;
      double s[63], w[63], *o = &t[pb.first * kPoleBlock];
      inv_sqrt_poles(kappa, K, s, w);
      for (int j = 0; j < K; ++j) {
        const int at = j < 31 ? j : kPoleBlock + j - 31;
        o[at] = s[j];
        o[at + 32] = w[j];
      }
    }
    return t;
  }();
  return table;
}

}  // namespace oakg
