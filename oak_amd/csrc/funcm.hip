// The matrix functions of M = I + C that the analysis needs, from its
// tridiagonal form M = Q T Q^T (N > 32), without eigenvectors:
//
//   R = M^-1/2                 (rrsqrt.F90:185; the transform is R Omega)
//   a = M^-1 b                 (rrsqrt.F90:142)
//   v = M^1/2 1 / |M^1/2 1|    (rrsqrt.F90:176-177)
//
// x^-1/2 on [1, kappa] is Zolotarev's best rational approximation in partial
// fractions, sum_j w_j / (x + s_j) with 31 poles -s_j < 0 (N. J. Higham,
// "Functions of Matrices", 2008, section 5.2; J. van den Eshof et al., Comput.
// Phys. Commun. 146, 2002; N. Hale, N. J. Higham and L. N. Trefethen, SIAM J.
// Numer. Anal. 46, 2008).  Its relative error is 5e-16 at kappa = 1e6 and
// grows to 1e-7 at 1e15, four orders below the eps kappa by which rounding C
// moves M^-1/2 in any case.  Then
//
//   T^-1/2 = sum_j w_j (T + s_j)^-1,  T^1/2 c = sum_j w_j (c - s_j (T + s_j)^-1 c)
//
// and each (T + s)^-1 is semiseparable: with the pivots gamma_0 = d_0 + s,
// gamma_i = d_i + s - e_{i-1}^2 / gamma_{i-1} and rho_i = -e_i / gamma_i,
//
//   G_kk = 1/gamma_k + rho_k^2 G_{k+1,k+1},   G_ik = rho_i G_{i+1,k}  (i < k).
//
// T >= I (M is I plus a positive semidefinite matrix), so every exact pivot is
// at least 1 + s: a pivot that rounding leaves below is set to it, as
// rrsqrt.F90:137 clamps the eigenvalues.  One lane per pole runs the two
// recurrences (about 60 cycles a row); a QL iteration with its ~1.1 N^2 plane
// rotations on the rows of Q, which this replaces, took 22 of the 45 ms of
// the eigensolve of 64 800 zones at N = 128.
#include <math.h>

#include <mutex>

#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"

namespace oakg {

namespace {

constexpr int kPoles = 31;    // lane 31 of the pole wave carries s = 0 (T itself)
constexpr int kBuckets = 25;  // kappa = 4, 16, ... 4^25

// [bucket][0: s, 1: w][pole]; pole 31: s = 0, w = 0
__device__ double g_poles[kBuckets][2][32];

// Poles and weights for [1, kappa], in extended precision.  With k =
// kappa^-1/2 the zeros and poles are -c_j, c_j = sc^2(j K' / 62) (modulus
// k' = sqrt(1 - k^2)), by the descending Landen transformation for the lower
// half and c_{62-j} = kappa / c_j for the upper one.
void zolotarev(long double kappa, double* s, double* w) {
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

std::mutex g_pole_mu;
bool g_pole_done[64] = {};

}  // namespace

// Fills the current device's table (once per device, before any launch).
hipError_t init_poles(int device) {
  std::lock_guard<std::mutex> lock(g_pole_mu);
  if (device >= 0 && device < 64 && g_pole_done[device]) return hipSuccess;
  static double host[kBuckets][2][32];
  long double kappa = 1.0L;
  for (int b = 0; b < kBuckets; ++b) {
    kappa *= 4.0L;
    zolotarev(kappa, host[b][0], host[b][1]);
  }
  const hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(g_poles), host, sizeof host);
  if (e == hipSuccess && device >= 0 && device < 64) g_pole_done[device] = true;
  return e;
}

// ---------------------------------------------------------------------------
// R, a and v of a zone, one workgroup (4 waves) per zone:
//   1. wave 0, one lane per pole: pivots, the diagonal of (T + s)^-1 and the
//      solves with Q^T b (s = 0) and Q^T 1, top down then bottom up; waves
//      1..3 meanwhile form the triangular factors T_b of the reflector
//      blocks (H_k0 ... H_k0+15 = I - V T_b V^T, compact WY, LAPACK dlarft)
//   2. F = T^-1/2 in 16 x 16 tiles in the accumulators, wave w holding tile
//      columns w (and NP/16 - 1 - w): the tiles off the diagonal are products
//      over the poles (MFMA, 8 steps) of row and column factors of the
//      semiseparable form relative to the tile edges; the diagonal tiles run
//      the recurrence
//   3. R = Q F Q^T, block by block from the last reflectors: with X = F V,
//      S = V^T X and P = T_b^T V^T,
//        F <- F - V T_b (X^T - S P) - X P,
//      each wave on its own tile columns (X through LDS), and [a, v] = Q [x, y]
//      along the way.  F stays symmetric; it is kept whole, since the MFMA
//      contracts over a tile's rows and the lower half alone would need the
//      transposed tiles.
// The MFMAs of step 3 are the bound (3456 of 16 x 16 x 4 per zone at NP = 128,
// 14.9 us on a CU); two zones share a CU (80 KB of LDS), three at NP = 64, so
// that one zone's pole recurrences run under another's MFMAs.
// DUAL (observation-space zones, dual.hip): F with the weights w / (1 + s),
// i.e. x -> 1 / (x + sqrt x), and y with w s / (1 + s), x -> 1 / (1 + sqrt x);
// v is left as Q y.  TR is the type R is stored in (float for the FP32 update
// of the mixed path).
// ---------------------------------------------------------------------------
template <int NP>
struct FuncLds {
  static constexpr int NB = NP / 16, LV = 18;
  union {
    struct {
      double a[NP * 32];  // rho, then the row factors alpha
      double g[NP * 32];  // G_kk, then the column factors beta
    } p;
    struct {
      double vb[2][NP * LV];  // V[r][j]: row r of reflector 16 b + j
      double x[NP * LV];      // X = F V
      double s[4][16 * 17];   // each wave's share of S = V^T X
      double g[2][16];        // V^T [x, y]
      double t[4][2][16];     // T_b V^T [x, y], per wave
    } m;
  };
  double tp[NB * 136];  // T_b, packed by columns (upper triangles)
  union {
    double dia[4][136];  // each wave's diagonal tile
    struct {
      double d[NP], e[NP];
      double gs[3][136];  // V^T V of waves 1..3
    } c;
  } w;
  double c[2][NP];  // Q^T b, Q^T 1; then x, y; then a, v
  int bucket;
};

// position of pole j of row r: 16-byte pairs swapped within the row, so that
// the operand reads (16 rows x 4 pairs) spread over the banks
__device__ __forceinline__ int pole_at(int r, int j) {
  return r * 32 + ((((j >> 1) ^ r) & 15) << 1) + (j & 1);
}

// eight consecutive poles 8 kk .. 8 kk + 7 of row r
__device__ __forceinline__ void load_poles(const double* arr, int r, int kk, double (&o)[8]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const double2 v = *reinterpret_cast<const double2*>(arr + r * 32 + ((((4 * kk + c) ^ r) & 15) << 1));
    o[2 * c] = v.x;
    o[2 * c + 1] = v.y;
  }
}

__device__ __forceinline__ double row_sum16(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x124>(v);
  v += dpp_d<0x128>(v);
  return v;
}

template <int NP, bool DUAL, typename TR>
__global__ __launch_bounds__(256, 2) void k_func(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                 const int64_t* __restrict__ sel_ptr,
                                                 double* __restrict__ qmat,
                                                 const double* __restrict__ dvec,
                                                 const double* __restrict__ evec,
                                                 double* __restrict__ vec, double* __restrict__ ampl,
                                                 unsigned* __restrict__ err, int likelihood) {
  using L = FuncLds<NP>;
  constexpr int NB = L::NB, LV = L::LV, TC = NB / 4, ER = NP / 16;
  __shared__ L S;
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;  // the zone is solved by the other pipeline
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane >> 4, lc = lane & 15;
  double* Vz = vec + (size_t)zl * 4 * NP;
  if (sel_ptr[z + 1] == sel_ptr[z]) {  // no observations: a = 0
    if (tid < NP) Vz[NP + tid] = 0.0;
    return;
  }
  double* V = qmat + (size_t)zl * NP * NP;
  if (tid < NP) {
    S.w.c.d[tid] = dvec[(size_t)zl * NP + tid];
    S.w.c.e[tid] = tid < NP - 1 ? evec[(size_t)zl * NP + tid] : 0.0;
    S.c[0][tid] = Vz[tid];
    S.c[1][tid] = Vz[2 * NP + tid];
  }
  lds_barrier();
  if (wave == 0) {
    // ---- pivots and solves, one lane per pole ----
    double nt = 0.0;  // Gershgorin bound of T
#pragma unroll
    for (int h = 0; h < NP / 64; ++h) {
      const int r = lane + 64 * h;
      nt = fmax(nt, fabs(S.w.c.d[r]) + fabs(S.w.c.e[r]) + (r > 0 ? fabs(S.w.c.e[r - 1]) : 0.0));
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) nt = fmax(nt, shfl_xor_d(nt, o));
    // smallest kappa = 4^(bucket+1) >= nt (nt < 2^ex)
    const int ex = (__double2hiint(nt) >> 20) - 1022;
    int bk = ((ex + 1) >> 1) - 1;
    bk = bk < 0 ? 0 : (bk > kBuckets - 1 ? kBuckets - 1 : bk);
    bk = __builtin_amdgcn_readfirstlane(bk);
    if (lane == 0) S.bucket = bk;
    if (lane < 32) {
      const double s = g_poles[bk][0][lane], sp1 = 1.0 + s;
      double wj = g_poles[bk][1][lane];
      if (DUAL) wj = wj * s / sp1;
      const double* cc = S.c[lane == 31 ? 0 : 1];
      double rho = 0.0, z1 = 0.0, ep = 0.0;
#pragma unroll 1
      for (int t = 0; t < NB; ++t) {
        double dv[16], ev[16], cv[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          dv[i] = S.w.c.d[16 * t + i];
          ev[i] = S.w.c.e[16 * t + i];
          cv[i] = cc[16 * t + i];
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const double gam = fmax(fma(ep, rho, dv[i] + s), sp1);
          const double inv = rcp_acc(gam);
          z1 = fma(rho, z1, cv[i]);
          const int at = pole_at(16 * t + i, lane);
          S.p.a[at] = inv;
          S.p.g[at] = z1 * inv;
          rho = -ev[i] * inv;
          ep = ev[i];
        }
      }
      double x = 0.0, G = 0.0, slog = 0.0, sinv = 0.0, sba = 0.0;
#pragma unroll 1
      for (int t = NB - 1; t >= 0; --t) {
        double iv[16], zi[16], ev[16], tv[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int at = pole_at(16 * t + i, lane);
          iv[i] = S.p.a[at];
          zi[i] = S.p.g[at];
          ev[i] = S.w.c.e[16 * t + i];
          tv[i] = S.c[1][16 * t + i];
        }
#pragma unroll
        for (int i = 15; i >= 0; --i) {
          const double r = -ev[i] * iv[i];
          G = fma(r * r, G, iv[i]);
          x = fma(r, x, zi[i]);
          const int at = pole_at(16 * t + i, lane);
          S.p.a[at] = r;
          S.p.g[at] = G;
          tv[i] = DUAL ? wj * x : wj * fma(-s, x, tv[i]);
          if (likelihood) {
            slog -= log(iv[i]);
            sinv += 1.0 - G;
            sba = fma(S.c[0][16 * t + i], x, sba);
          }
          if (lane == 31) S.c[0][16 * t + i] = x;
        }
        // sums over the poles: lanes 0..15 keep rows 0..7, lanes 16..31 rows 8..15
        const bool up = lane >= 16;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const double give = up ? tv[i] : tv[i + 8], keep = up ? tv[i + 8] : tv[i];
          tv[i] = row_sum16(keep + shfl_xor_d(give, 16));
        }
        if (lc == 0) {
#pragma unroll
          for (int i = 0; i < 8; ++i) S.c[1][16 * t + (up ? 8 : 0) + i] = tv[i];
        }
      }
      if (likelihood && lane == 31) {  // log det M, sum (1 - 1/mu) and b^T a
        Vz[3 * NP] = slog;
        Vz[3 * NP + 1] = sinv;
        Vz[3 * NP + 2] = sba;
      }
    }
  } else {
    // ---- T_b of the reflector blocks ----
    for (int b = wave - 1; b < NB; b += 3) {
      const int k = 16 * b + lc;
      const double* src = V + (size_t)k * NP;
      d4 g = {0.0, 0.0, 0.0, 0.0};
      for (int k0 = 4 * b; k0 < NP / 4; k0 += 4) {
        double xv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int r = 4 * (k0 + u) + lr;
          xv[u] = (k < NP - 2 && r > k) ? src[r] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) g = mfma_f64(xv[u], xv[u], g);
      }
      const double tau = (lane < 16 && k < NP - 2) ? src[k] : 0.0;
      double* gs = S.w.c.gs[wave - 1];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (lr + 4 * r <= lc) gs[lc * (lc + 1) / 2 + lr + 4 * r] = g[r];
      __builtin_amdgcn_wave_barrier();
      // T_b[j][j] = tau_j, T_b[0:j, j] = -tau_j T_b[0:j, 0:j] (V^T V)[0:j, j]
      double tr[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        asm volatile("" ::: "memory");  // column by column, not all loads at once
        double sm = 0.0;
#pragma unroll
        for (int q = 0; q < j; ++q) sm = fma(tr[q], gs[j * (j + 1) / 2 + q], sm);
        const double tj = readlane_d(tau, j);
        tr[j] = lane < j ? -tj * sm : (lane == j ? tj : 0.0);
        if (lane <= j) S.tp[b * 136 + j * (j + 1) / 2 + lane] = tr[j];
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  lds_barrier();
  // ---- F = T^-1/2 ----
  const int J0 = wave, J1 = NB - 1 - wave;  // tile columns (TC = 1: J0 only)
  d4 f[TC][NB];
  double wq[8];
  {
    const int bk = S.bucket;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      wq[q] = g_poles[bk][1][8 * lr + q];
      if (DUAL) wq[q] = wq[q] / (1.0 + g_poles[bk][0][8 * lr + q]);
    }
  }
  // diagonal tiles: lane (lr, lc) runs column lc up from its diagonal entry
  // for its eight poles
#pragma unroll
  for (int jj = 0; jj < TC; ++jj) {
    const int J = jj ? J1 : J0;
    double g[8];
    load_poles(S.p.g, 16 * J + lc, lr, g);
#pragma unroll
    for (int q = 0; q < 8; ++q) g[q] *= wq[q];
    double* dia = S.w.dia[wave];
#pragma unroll 1
    for (int i = 15; i >= 0; --i) {
      double r[8];
      load_poles(S.p.a, 16 * J + i, lr, r);
#pragma unroll
      for (int q = 0; q < 8; ++q) g[q] *= i < lc ? r[q] : 1.0;
      double sm = ((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7]));
      sm += shfl_xor_d(sm, 16);
      sm += shfl_xor_d(sm, 32);
      if (lr == 0 && i <= lc) dia[lc * (lc + 1) / 2 + i] = sm;
    }
    __builtin_amdgcn_wave_barrier();
    d4 fd;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = lr + 4 * r, hi = i > lc ? i : lc, lo = i > lc ? lc : i;
      fd[r] = dia[hi * (hi + 1) / 2 + lo];
    }
#pragma unroll
    for (int I = 0; I < NB; ++I)
      if (I == J) f[jj][I] = fd;
    __builtin_amdgcn_wave_barrier();
  }
  lds_barrier();
  // alpha_i = rho_i ... rho_{last row of the tile}, beta_k = G_kk rho_{first} ... rho_{k-1}
  if (tid < 32 * NB) {
    const int t = tid >> 5, j = tid & 31;
    double r[16], g[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int at = pole_at(16 * t + i, j);
      r[i] = S.p.a[at];
      g[i] = S.p.g[at];
    }
    double pi = 1.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      g[i] *= pi;
      pi *= r[i];
    }
#pragma unroll
    for (int i = 14; i >= 0; --i) r[i] *= r[i + 1];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int at = pole_at(16 * t + i, j);
      S.p.a[at] = r[i];
      S.p.g[at] = g[i];
    }
  }
  lds_barrier();
  {
    double B[TC][8];
#pragma unroll
    for (int jj = 0; jj < TC; ++jj) {  // tiles above the diagonal, upwards
      load_poles(S.p.g, 16 * (jj ? J1 : J0) + lc, lr, B[jj]);
#pragma unroll
      for (int q = 0; q < 8; ++q) B[jj][q] *= wq[q];
    }
#pragma unroll
    for (int I = NB - 2; I >= 0; --I) {
      asm volatile("" ::: "memory");
      double al[8], edge[8];
      load_poles(S.p.a, 16 * I + lc, lr, al);
      load_poles(S.p.a, 16 * I, lr, edge);
#pragma unroll
      for (int jj = 0; jj < TC; ++jj)
        if (I < (jj ? J1 : J0)) {
          d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            acc = mfma_f64(al[q], B[jj][q], acc);
            B[jj][q] *= edge[q];
          }
          f[jj][I] = acc;
        }
    }
#pragma unroll
    for (int jj = 0; jj < TC; ++jj) {  // tiles below the diagonal, downwards
      load_poles(S.p.a, 16 * (jj ? J1 : J0) + lc, lr, B[jj]);
#pragma unroll
      for (int q = 0; q < 8; ++q) B[jj][q] *= wq[q];
    }
#pragma unroll
    for (int I = 1; I < NB; ++I) {
      asm volatile("" ::: "memory");
      double be[8], edge[8];
      load_poles(S.p.g, 16 * I + lc, lr, be);
      load_poles(S.p.a, 16 * I, lr, edge);
#pragma unroll
      for (int jj = 0; jj < TC; ++jj)
        if (I > (jj ? J1 : J0)) {
          d4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            acc = mfma_f64(be[q], B[jj][q], acc);
            B[jj][q] *= edge[q];
          }
          f[jj][I] = acc;
        }
    }
  }
  // ---- R = Q F Q^T, [a, v] = Q [x, y] ----
  // thread t moves reflector pj = t / 16 of a block, rows pr + 16 e
  const int pj = tid >> 4, pr = tid & 15;
  double pf[ER];
  auto load_block = [&](int b) {
    const int k = 16 * b + pj;
    const double* src = V + (size_t)k * NP + pr;
#pragma unroll
    for (int e = 0; e < ER; ++e) pf[e] = (k < NP - 2 && pr + 16 * e > k) ? src[16 * e] : 0.0;
  };
  load_block(NB - 1);
  lds_barrier();  // the pole arrays are read
#pragma unroll 1
  for (int b = NB - 1; b >= 0; --b) {
    double* vb = S.m.vb[b & 1];
#pragma unroll
    for (int e = 0; e < ER; ++e) vb[(pr + 16 * e) * LV + pj] = pf[e];
    if (b > 0) load_block(b - 1);
    lds_barrier();
    {  // V^T [x, y]
      double g0 = 0.0, g1 = 0.0;
#pragma unroll
      for (int e = 0; e < ER; ++e) {
        const int r = pr + 16 * e;
        const double vv = vb[r * LV + pj];
        g0 = fma(vv, S.c[0][r], g0);
        g1 = fma(vv, S.c[1][r], g1);
      }
      g0 = row_sum16(g0);
      g1 = row_sum16(g1);
      if (pr == 0) {
        S.m.g[0][pj] = g0;
        S.m.g[1][pj] = g1;
      }
    }
    d4 y[TC], sp = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int jj = 0; jj < TC; ++jj) y[jj] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int I = 0; I < NB; ++I)
      if (I >= b) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double vv = vb[(16 * I + 4 * q + lr) * LV + lc];
#pragma unroll
          for (int jj = 0; jj < TC; ++jj) y[jj] = mfma_f64(vv, f[jj][I][q], y[jj]);
        }
      }
#pragma unroll
    for (int jj = 0; jj < TC; ++jj) {
      const int J = jj ? J1 : J0;
#pragma unroll
      for (int r = 0; r < 4; ++r) S.m.x[(16 * J + lc) * LV + lr + 4 * r] = y[jj][r];
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int jj = 0; jj < TC; ++jj) {
      const int J = jj ? J1 : J0;
      if (J >= b) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int at = (16 * J + 4 * q + lr) * LV + lc;
          sp = mfma_f64(S.m.x[at], vb[at], sp);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) S.m.s[wave][(lr + 4 * r) * 17 + lc] = sp[r];
    lds_barrier();
    const double* tp = S.tp + b * 136;
    double tt[4], tn[4], sa[4];  // T_b^T, T_b and S as A operands
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int k = 4 * q + lr, hi = k > lc ? k : lc, lo = k > lc ? lc : k;
      const double tv = tp[hi * (hi + 1) / 2 + lo];
      tt[q] = k <= lc ? tv : 0.0;
      tn[q] = lc <= k ? tv : 0.0;
      const int at = lc * 17 + k;
      sa[q] = (S.m.s[0][at] + S.m.s[1][at]) + (S.m.s[2][at] + S.m.s[3][at]);
    }
    d4 qv[TC], pv[TC];
#pragma unroll
    for (int jj = 0; jj < TC; ++jj) {
      const int J = jj ? J1 : J0;
      pv[jj] = d4{0.0, 0.0, 0.0, 0.0};
      if (J >= b) {
        d4 s2 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q) pv[jj] = mfma_f64(tt[q], vb[(16 * J + lc) * LV + 4 * q + lr], pv[jj]);
#pragma unroll
        for (int q = 0; q < 4; ++q) s2 = mfma_f64(sa[q], pv[jj][q], s2);
#pragma unroll
        for (int q = 0; q < 4; ++q) y[jj][q] -= s2[q];
      }
      qv[jj] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q) qv[jj] = mfma_f64(tn[q], y[jj][q], qv[jj]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        qv[jj][q] = -qv[jj][q];
        pv[jj][q] = -pv[jj][q];
      }
    }
    {  // [x, y] <- [x, y] - V (T_b V^T [x, y])
      double* tw = S.m.t[wave][0];
      if (lane < 32) {
        double sm = 0.0;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const double tv = tp[k * (k + 1) / 2 + (lc <= k ? lc : k)];
          sm = fma(lc <= k ? tv : 0.0, S.m.g[lr][k], sm);
        }
        tw[lane] = sm;
      }
      __builtin_amdgcn_wave_barrier();
      if (tid < 2 * NP) {
        const int vq = tid / NP, r = tid % NP;
        double sm = S.c[vq][r];
#pragma unroll
        for (int k = 0; k < 16; ++k) sm = fma(-vb[r * LV + k], tw[16 * vq + k], sm);
        S.c[vq][r] = sm;
      }
    }
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      if (I >= b) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double vv = vb[(16 * I + lc) * LV + 4 * q + lr];
#pragma unroll
          for (int jj = 0; jj < TC; ++jj) f[jj][I] = mfma_f64(vv, qv[jj][q], f[jj][I]);
        }
      }
      if ((TC > 1 ? J1 > J0 ? J1 : J0 : J0) >= b) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double xv = S.m.x[(16 * I + lc) * LV + 4 * q + lr];
#pragma unroll
          for (int jj = 0; jj < TC; ++jj)
            if ((jj ? J1 : J0) >= b) f[jj][I] = mfma_f64(xv, pv[jj][q], f[jj][I]);
        }
      }
    }
  }
  TR* R = reinterpret_cast<TR*>(V);  // every reflector was read before the last barrier
#pragma unroll
  for (int jj = 0; jj < TC; ++jj)
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        R[(size_t)(16 * I + lr + 4 * r) * NP + 16 * (jj ? J1 : J0) + lc] = (TR)f[jj][I][r];
  lds_barrier();
  if (tid < NP) {
    double nv = 0.0;
#pragma unroll
    for (int h = 0; h < NP / 64; ++h) {
      const double vv = S.c[1][lane + 64 * h];
      nv = fma(vv, vv, nv);
    }
    nv = wave_sum_fast(nv);
    const double ar = S.c[0][tid], vr = S.c[1][tid];
    Vz[NP + tid] = ar;
    Vz[2 * NP + tid] = DUAL ? vr : vr / sqrt(nv);
    if (ampl && tid < N) ampl[(size_t)z * N + tid] = ar;
    if (ar != ar) atomicOr(err, OAKG_DERR_NAN);
  }
}

// R = Y Y^T (and the likelihood's log det M, sum (1 - 1/mu) and b^T a) from
// the Y = U diag(mu^-1/4) and mu of the Jacobi option, so that one form
// reaches the transform.
template <int NP, typename TR>
__global__ __launch_bounds__(256) void k_yyt(int64_t z0, const int32_t* __restrict__ zorder,
                                             const int64_t* __restrict__ sel_ptr,
                                             double* __restrict__ ymat, double* __restrict__ vec) {
  constexpr int LD = NP + 1, NB = NP / 16;
  __shared__ double Y[NP * LD];
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;
  if (sel_ptr[z + 1] == sel_ptr[z]) return;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane >> 4, lc = lane & 15;
  double* Yz = ymat + (size_t)zl * NP * NP;
  double* Vz = vec + (size_t)zl * 4 * NP;
  double slog = 0.0, sinv = 0.0, sba = 0.0;
  if (wave == 0) {
    for (int k = lane; k < NP; k += 64) {
      const double mu = Vz[3 * NP + k];
      slog += log(mu);
      sinv += 1.0 - 1.0 / mu;
      sba = fma(Vz[k], Vz[NP + k], sba);
    }
    slog = wave_sum_fast(slog);
    sinv = wave_sum_fast(sinv);
    sba = wave_sum_fast(sba);
  }
  for (int e = tid; e < NP * NP; e += 256) Y[(e / NP) * LD + e % NP] = Yz[e];
  __syncthreads();
  TR* R = reinterpret_cast<TR*>(Yz);
  for (int t = wave; t < NB * NB; t += 4) {
    const int I = t / NB, J = t % NB;
    d4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int k = 0; k < NP; k += 4)
      acc = mfma_f64(Y[(16 * I + lc) * LD + k + lr], Y[(16 * J + lc) * LD + k + lr], acc);
#pragma unroll
    for (int r = 0; r < 4; ++r) R[(size_t)(16 * I + lr + 4 * r) * NP + 16 * J + lc] = (TR)acc[r];
  }
  if (tid == 0) {
    Vz[3 * NP] = slog;
    Vz[3 * NP + 1] = sinv;
    Vz[3 * NP + 2] = sba;
  }
}

// The reduction (wide256.hip) and the functions of T for a chunk at NP = 64
// or 128 (dual: the observation-space zones).
void launch_func(int NP, const ChunkArgs& A, bool dual, hipStream_t st) {
  const dim3 g(A.nzc), b(256);
  const int like = A.mode == 2;
#define OAK_FUNC(P, D, TR)                                                                      \
  hipLaunchKernelGGL((k_func<P, D, TR>), g, b, 0, st, A.z0, A.zorder, A.N, A.sel_ptr, A.ymat,   \
                     A.dvec, A.evec, A.vec, A.ampl, A.err, like)
  if (NP == 64) {
    launch_tridiag_lower64(A, dual ? -1 : A.N, st);
    if (dual)
      OAK_FUNC(64, true, double);
    else
      OAK_FUNC(64, false, double);
  } else {
    launch_tridiag_lower128(A, A.N, st);
    if (A.prec == 1)
      OAK_FUNC(128, false, float);
    else
      OAK_FUNC(128, false, double);
  }
#undef OAK_FUNC
}

void launch_yyt(int NP, const ChunkArgs& A, hipStream_t st) {
  const dim3 g(A.nzc), b(256);
#define OAK_YYT(P, TR) \
  hipLaunchKernelGGL((k_yyt<P, TR>), g, b, 0, st, A.z0, A.zorder, A.sel_ptr, A.ymat, A.vec)
  if (NP == 64)
    OAK_YYT(64, double);
  else if (A.prec == 1)
    OAK_YYT(128, float);
  else
    OAK_YYT(128, double);
#undef OAK_YYT
}

}  // namespace oakg
