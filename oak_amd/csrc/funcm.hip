// The matrix functions of M = I + C that the analysis needs, from its
// tridiagonal form M = Q T Q^T, without eigenvectors:
//
//   R = M^-1/2                 (rrsqrt.F90:185; the transform is R Omega)
//   a = M^-1 b                 (rrsqrt.F90:142)
//   v = M^1/2 1 / |M^1/2 1|    (rrsqrt.F90:176-177)
//
// x^-1/2 on [1, kappa] is Zolotarev's best rational approximation in partial
// fractions, sum_j w_j / (x + s_j) with poles -s_j < 0 (N. J. Higham, "Functions
// of Matrices", 2008, section 5.2; J. van den Eshof et al., Comput. Phys. Commun.
// 146, 2002), for kappa above a bound of T's spectrum: 31 poles, a lane each, up
// to kappa = 2^20, 63 in two blocks one after the other up to 2^44, to 4.3e-16
// either way (poles.hpp).  Then
//
//   T^-1/2 = sum_j w_j (T + s_j)^-1,  T^1/2 c = sum_j w_j (c - s_j (T + s_j)^-1 c)
//
// and each G = (T + s)^-1 is semiseparable.  Eliminating from both ends to the
// middle row h = NP/2 - 1, with the pivots gamma_0 = d_0 + s, gamma_i = d_i + s
// - e_{i-1}^2 / gamma_{i-1} above it, the same from the bottom below it, and
// tau_i = -e / gamma_i (e the coupling of row i towards the middle),
//
//   G_hh = 1 / (gamma_h - e_h^2 / gamma_{h+1}),  and outwards
//   G_ii = 1/gamma_i + tau_i^2 G_mm,  G_ik = tau_i G_mk
//
// for m the neighbour of i towards the middle and every k at or beyond m.
// T >= I (M is I plus a positive semidefinite matrix), so every exact pivot is
// at least 1 + s: a pivot that rounding leaves below is set to it.  One lane per
// pole and half runs the recurrences, NP/2 rows in and NP/2 rows out; a QL
// iteration with its ~1.1 N^2 plane rotations on the rows of Q, which this
// replaces, took 22 of the 45 ms of the eigensolve of 64 800 zones at N = 128.
//
// Above kappa = 2^44 rounding C has moved T's small eigenvalues by a part of 1 and
// more.  A zone with fewer such precise observations than members can be
// indefinite, bounded pivots are no bound on G then (Sa came out up to 1e266 off),
// and only the eigenvalues can be cut off at 1 as rrsqrt.F90:137 does: these zones
// take QL (ql_functions) in the kernel that meets them.
#include <math.h>
#include <stddef.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"
#include "poles.hpp"

namespace oakg {

// ---------------------------------------------------------------------------
// Zones beyond the poles: eigenvalues and eigenvectors of T by implicit QL
// (A. Dubrulle, R. S. Martin and J. H. Wilkinson, Numer. Math. 12, 1968), a sweep's
// rotations by the last wave while a thread per row applies the sweep before.
// Called by the NT threads of a workgroup; Z: NP x NP in LDS or global memory, row k
// of it eigenvector k.
// T comes with its rows in reverse: the reduction leaves the strongly observed
// directions in the first rows, and QL wants the large entries last (with them first,
// the small eigenvalues came out ten times less accurate).
// Negligible couplings are those below the rounding of the largest entries, too: with
// fewer observations than members the reduction leaves no others after some rows, and
// QL is soon done.  Bound by the chain of the 1.1 NP^2 rotations otherwise, and at N > 64
// by the rows of Z through the caches.  4096 zones of N = 128 with 256 observations of
// a ten millionth of the spread: 29 ms with the reduction, with 32 of them 6.1 (two
// blocks of poles 5.5, one 2.2; QL over the lanes of a wave, a zone each, took 9.5 and
// 3.5 in all).
// ---------------------------------------------------------------------------
template <int NP>
struct QlLds {
  double d[NP], e[NP];     // T, last row first (e_i couples i and i + 1); then the weights of F in e
  double c[2][NP];         // cosines of two sweeps; then Z^T u in c[0] and s[0]
  double u[2][NP];         // Q^T b, Q^T 1; then x, y
  double s[2][NP];         // sines
  int range[2][2];         // the sweeps' first and last row; -1: no sweep
};

// Largest |d| + |e| of T below 2^ex (of a finite T; 1025 for infinities).
__device__ __forceinline__ int exponent_above(double nt) { return (__double2hiint(nt) >> 20) - 1022; }

// The next sweep's rotations (one wave, every lane the same numbers).
template <int NP>
__device__ __forceinline__ void ql_sweep(QlLds<NP>& S, double tiny, int buf) {
  const int lane = threadIdx.x & 63;
  // the first coupling lo that is not negligible, and the first after it that is
  int lo = -1, hi = -1;
  for (int b = 0; b < NP && hi < 0; b += 64) {
    const int i = b + lane;
    const bool live = i < NP - 1 && fabs(S.e[i < NP ? i : 0]) >
                                        fmax(0x1p-53 * (fabs(S.d[i < NP ? i : 0]) + fabs(S.d[i < NP - 1 ? i + 1 : 0])), tiny);
    const unsigned long long on = __ballot(live);
    unsigned long long off = ~on;
    if (lo < 0) {
      if (on == 0) continue;
      const int t = __ffsll((long long)on) - 1;
      lo = b + t;
      off &= ~((2ull << t) - 1ull);
    }
    if (off != 0) hi = b + __ffsll((long long)off) - 1;
  }
  if (lo >= 0) {
    const double dl = S.d[lo], el = S.e[lo];
    double dn = S.d[hi], di = S.d[hi - 1], ei = S.e[hi - 1];  // rows i + 1 and i
    double g = (S.d[lo + 1] - dl) / (2.0 * el);
    g = dn - dl + el / (g + copysign(sqrt(fma(g, g, 1.0)), g));
    double s = 1.0, c = 1.0, p = 0.0;
    for (int i = hi - 1; i >= lo; --i) {
      const int nx = i > lo ? i - 1 : lo;
      const double dx = S.d[nx], ex = S.e[nx];  // the next row's, ahead of the chain
      const double f = s * ei, b = c * ei, hh = fma(f, f, g * g);
      const bool turns = hh > 0x1p-900;  // else no rotation
      const double rn = rsqrt_acc(turns ? hh : 1.0);
      s = turns ? f * rn : 0.0;
      c = turns ? g * rn : 1.0;
      S.e[i + 1] = turns ? hh * rn : 0.0;
      g = dn - p;
      const double q = fma(di - g, s, 2.0 * c * b);
      p = s * q;
      S.d[i + 1] = g + p;
      g = fma(c, q, -b);
      S.c[buf][i] = c;
      S.s[buf][i] = s;
      dn = di;
      di = dx;
      ei = ex;
    }
    S.d[lo] = dl - p;
    S.e[lo] = g;
    S.e[hi] = 0.0;
  }
  if (lane == 0) {
    S.range[buf][0] = lo;
    S.range[buf][1] = hi;
  }
}

template <int NP, int NT, bool DUAL>
__device__ __forceinline__ void ql_functions(QlLds<NP>& S, double nt, double* Z) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const bool leads = wave == NT / 64 - 1;
  if (tid < NP)
    for (int k = 0; k < NP; ++k) Z[(size_t)k * NP + tid] = k == NP - 1 - tid ? 1.0 : 0.0;
  // couplings that are rounding of the largest entries: with as many members as
  // observations and more the reduction leaves only those after some rows
  const double tiny = 0x1p-53 * nt;
  if (leads) ql_sweep<NP>(S, tiny, 0);
  __syncthreads();
  // two sweeps an eigenvalue are usual; the bound ends any other case
#pragma unroll 1
  for (int sweep = 0; sweep < 40 * NP; ++sweep) {
    const int buf = sweep & 1, lo = S.range[buf][0], hi = S.range[buf][1];
    if (lo < 0) break;
    if (leads) ql_sweep<NP>(S, tiny, buf ^ 1);
    if (tid < NP) {
      // eight rows at a time, with the next eight (clamped to lo) in flight
      constexpr int Q = 8;
      auto at = [&](int i) { return i > lo ? i : lo; };
      double zc = Z[(size_t)hi * NP + tid], zi[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) zi[q] = Z[(size_t)at(hi - 1 - q) * NP + tid];
#pragma unroll 1
      for (int i0 = hi - 1; i0 >= lo; i0 -= Q) {
        double zn[Q], c[Q], s[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          zn[q] = Z[(size_t)at(i0 - Q - q) * NP + tid];
          c[q] = S.c[buf][at(i0 - q)];
          s[q] = S.s[buf][at(i0 - q)];
        }
        if (i0 - Q + 1 >= lo) {
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            Z[(size_t)(i0 - q + 1) * NP + tid] = fma(s[q], zi[q], c[q] * zc);
            zc = fma(c[q], zi[q], -s[q] * zc);
          }
        } else {
#pragma unroll
          for (int q = 0; q < Q; ++q)
            if (i0 - q >= lo) {
              Z[(size_t)(i0 - q + 1) * NP + tid] = fma(s[q], zi[q], c[q] * zc);
              zc = fma(c[q], zi[q], -s[q] * zc);
            }
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) zi[q] = zn[q];
      }
      Z[(size_t)lo * NP + tid] = zc;
    }
    __syncthreads();
  }
  __syncthreads();
  // Z^T u, a wave per eigenvector, times the functions of mu = max(lambda, 1)
#pragma unroll 1
  for (int k = wave; k < NP; k += NT / 64) {
    double t0 = 0.0, t1 = 0.0;
    for (int r = lane; r < NP; r += 64) {
      const double zr = Z[(size_t)k * NP + r];
      t0 = fma(zr, S.u[0][r], t0);
      t1 = fma(zr, S.u[1][r], t1);
    }
    t0 = wave_sum_fast(t0);
    t1 = wave_sum_fast(t1);
    const double mu = S.d[k] < 1.0 ? 1.0 : S.d[k], sq = sqrt(mu);
    if (lane == 0) {
      S.c[0][k] = t0 / mu;
      S.s[0][k] = DUAL ? t1 / (1.0 + sq) : t1 * sq;
      S.e[k] = DUAL ? 1.0 / (mu + sq) : 1.0 / sq;
    }
  }
  __syncthreads();
  if (tid < NP) {
    double x = 0.0, y = 0.0;
    for (int k = 0; k < NP; ++k) {
      const double zk = Z[(size_t)k * NP + tid];
      x = fma(zk, S.c[0][k], x);
      y = fma(zk, S.s[0][k], y);
    }
    S.u[0][tid] = x;
    S.u[1][tid] = y;
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// R, a and v of a zone, one workgroup per zone, NP/16 waves:
//   1. wave 0, one lane per pole: pivots, the diagonal of (T + s)^-1 and the
//      solves with Q^T b (s = 0) and Q^T 1, top down then bottom up; the other
//      waves meanwhile form the triangular factors T_b of the reflector
//      blocks (H_k0 ... H_k0+15 = I - V T_b V^T, compact WY, LAPACK dlarft)
//   2. F = T^-1/2 in 16 x 16 tiles in the accumulators, each wave holding a
//      tile column: the tiles off the diagonal are products over the poles
//      (MFMA, 8 steps) of row and column factors of the semiseparable form
//      relative to the tile edges; the diagonal tiles run the recurrence
//   3. R = Q F Q^T, block by block from the last reflectors: with X = F V,
//      S = V^T X and P = T_b^T V^T,
//        F <- F - V T_b (X^T - S P) - X P,
//      each wave on its own tile column (X through LDS), and [a, v] = Q [x, y]
//      along the way.  F stays symmetric; it is kept whole, since the MFMA
//      contracts over a tile's rows and the lower half alone would need the
//      transposed tiles.
// The MFMAs of step 3 are the bound (3456 of 16 x 16 x 4 per zone at NP = 128,
// 23 us on a CU at 2.4 GHz); two zones of 8 waves share a CU (79 KB of LDS,
// 128 registers a lane), four at NP = 64, so that one zone's pole recurrences
// and barriers run under another's MFMAs.  Measured 60 us per zone and CU at
// NP = 128, 15 us at NP = 64 (8192 zones); two tile columns on each of four
// waves (256 registers) spilled and took 79 us, pivots from one end 66 us.
// DUAL (observation-space zones, dual.hip): F with the weights w / (1 + s),
// i.e. x -> 1 / (x + sqrt x), and y with w s / (1 + s), x -> 1 / (1 + sqrt x);
// v is left as Q y.  At NP = 128, R 1 and R v in slots 0 and 3 of vec.  TR is the type R is stored in (float for the FP32 update
// of the mixed path).
// ---------------------------------------------------------------------------
template <int NP>
struct FuncLds {
  static constexpr int NB = NP / 16, LV = 18;
  union {
    // rows in the order of the elimination: the upper half downwards, then the
    // lower half upwards (step_row)
    struct {
      double a[NP * 32];  // tau, then alpha
      double g[NP * 32];  // G_ii, then beta
      double d[NP];       // d; then G_hh of the poles
      double e[NP];       // coupling towards the middle
      double c[2][NP];    // Q^T b, Q^T 1; then x, y
    } p;
    struct {
      double vb[2][NP * LV];  // V[r][j]: row r of reflector 16 b + j
      double x[NP * LV];      // X = F V
      double s[NB][136];      // each wave's share of S = V^T X, packed
      double sf[16 * 17];     // S
      double g[2][16];        // V^T [x, y]
      double t[2][16];        // T_b V^T [x, y]
    } m;
    QlLds<NP> q;
  };
  double tp[NB * 136];  // T_b, packed by columns (upper triangles)
  double c[2][NP];      // x, y; then a, v
  double bound;         // of T's spectrum
  int first, count;     // the blocks of poles; count 0: QL
};

// place of row r in the elimination order, and back
template <int NP>
__device__ __forceinline__ int step_row(int r) {
  return r < NP / 2 ? r : NP / 2 + NP - 1 - r;
}

// position of pole j of row r (of that order): 16-byte pairs swapped within the row, so that
// the operand reads (16 rows x 4 pairs) spread over the banks
__device__ __forceinline__ int pole_at(int r, int j) {
  return r * 32 + ((((j >> 1) ^ r) & 15) << 1) + (j & 1);
}

// four consecutive poles 4 k4 .. 4 k4 + 3 of row r
__device__ __forceinline__ void load_poles4(const double* arr, int r, int k4, double (&o)[4]) {
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const double2 v = *reinterpret_cast<const double2*>(arr + r * 32 + ((((2 * k4 + c) ^ r) & 15) << 1));
    o[2 * c] = v.x;
    o[2 * c + 1] = v.y;
  }
}

// DEEP false: a zone of one block of poles (else false is returned); true: one of two
// or of none.
template <int NP, bool DUAL, typename TR, bool DEEP>
__device__ __forceinline__ bool func_zone(FuncLds<NP>& S, int zl, int64_t z, int N, int64_t cnt_obs,
                                          const double* __restrict__ ptab, double* __restrict__ qmat,
                                          const double* __restrict__ dvec,
                                          const double* __restrict__ evec,
                                          double* __restrict__ mat, double* __restrict__ vec,
                                          double* __restrict__ ampl, unsigned* __restrict__ err) {
  using L = FuncLds<NP>;
  constexpr int NB = L::NB, LV = L::LV;
  constexpr int TPR = NP / 4, ER = 4;  // threads per reflector of a block, rows of each
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane >> 4, lc = lane & 15;
  double* Vz = vec + (size_t)zl * 4 * NP;
  double* V = qmat + (size_t)zl * NP * NP;
  // order of M (the rest is the identity): the tiles and reflector blocks that
  // reach it take part
  const int n = DUAL ? (int)cnt_obs : N;
  const int nt = (n + 15) >> 4, nblk = n > 2 ? (n + 13) >> 4 : 0;
  auto load_t = [&]() {
    if (tid < NP) {
      const int k = step_row<NP>(tid);
      S.p.d[k] = dvec[(size_t)zl * NP + tid];
      S.p.e[k] = evec[(size_t)zl * NP + (tid < NP / 2 ? tid : tid - 1)];
      S.p.c[0][k] = Vz[tid];
      S.p.c[1][k] = Vz[2 * NP + tid];
    }
  };
  load_t();
  lds_barrier();
  // F = T^-1/2, tile column J (waves w and w + 4 share a SIMD: the
  // columns J and NB - 1 - J, whose updates add up alike).  The columns of the
  // lower half see the rows mirrored: f[I] is tile row I or NB - 1 - I, so that
  // I < Js lie outside the wave's own tile, Js < I < NB/2 towards the middle
  // and the rest beyond it
  const int J = wave < NB / 2 ? wave : NB + NB / 2 - 1 - wave;
  const bool low = J >= NB / 2;
  const int Js = low ? NB - 1 - J : J;
  auto row_of = [&](int I) { return low ? NB - 1 - I : I; };
  // place of tile row r in the pole arrays (elimination order)
  auto tile_of = [&](int r) { return r < NB / 2 ? r : NB / 2 + NB - 1 - r; };
  d4 f[NB];
  double* Fz = mat + (size_t)zl * NP * NP;  // M is no longer needed
#pragma unroll 1
  for (int batch = 0;; ++batch) {
    if (wave == 0) {
      // ---- pivots and solves, one lane per pole ----
      int blk = 0, cnt = 1;
      if (batch == 0) {
        double nt = 0.0;  // Gershgorin bound of T
#pragma unroll
        for (int h = 0; h < NP / 64; ++h) {
          const int k = lane + 64 * h;  // k's outer neighbour couples through e of k - 1
          nt = fmax(nt, fabs(S.p.d[k]) + fabs(S.p.e[k]) + (k % (NP / 2) ? fabs(S.p.e[k - 1]) : 0.0));
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) nt = fmax(nt, shfl_xor_d(nt, o));
        const int ex = __builtin_amdgcn_readfirstlane(exponent_above(nt));
        const PoleBlocks pb = pole_blocks(ex > 1024 ? 0 : ex);  // infinities end as NaN in a
        blk = pb.first;
        cnt = pb.count;
        if (lane == 0) {
          S.bound = nt;
          S.first = blk;
          S.count = cnt;
        }
        if (!DEEP && cnt != 1) cnt = 0;
      } else {
        blk = __builtin_amdgcn_readfirstlane(S.first + batch);
      }
      if (cnt != 0) {
        // lanes 0..31 rows 0 .. NP/2 - 1 downwards, lanes 32..63 the rest upwards
        const int j = lane & 31;
        const bool bot = lane >= 32;
        const bool tl = j == 31 && batch == 0;  // the lane of T itself
        const double s = ptab[blk * kPoleBlock + j], sp1 = 1.0 + s;
        double wj = ptab[blk * kPoleBlock + 32 + j];
        if (DUAL) wj = wj * s / sp1;
        const int h0 = bot ? NP / 2 : 0;
        const double* dd = S.p.d + h0;
        const double* ee = S.p.e + h0;
        double* cc = S.p.c[tl ? 0 : 1] + h0;  // the lane's right-hand side
        double* c1 = S.p.c[1] + h0;
        double* aa = S.p.a + h0 * 32;
        double* gg = S.p.g + h0 * 32;
        // position of the lane's pole in the row of step 16 t + i (i constant)
        auto at = [&](int t, int i) { return (16 * t + i) * 32 + ((j & ~1) ^ (2 * i)) + (j & 1); };
        double q = 0.0, z1 = 0.0, tau = 0.0, e2 = 0.0;
#pragma unroll 1
        for (int t = 0; t < NB / 2; ++t) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            asm volatile("" ::: "memory");  // the reads of eight rows at a time
            double dv[8], ev[8], cv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const int k = 16 * t + 8 * h + i;
              dv[i] = dd[k];
              ev[i] = ee[k];
              cv[i] = cc[k];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              q = rcp_acc(fmax(fma(-e2, q, dv[i] + s), sp1));
              z1 = fma(tau, z1, cv[i]);
              aa[at(t, 8 * h + i)] = q;
              gg[at(t, 8 * h + i)] = z1 * q;
              tau = -ev[i] * q;
              e2 = ev[i] * ev[i];
            }
          }
        }
        // the middle: q, z1 of rows h (top lanes) and h + 1 (bottom lanes);
        // 1 / G_hh = gamma_h - e_h^2 / gamma_{h+1}, x_h = G_hh (z_h + tau_{h+1} z_{h+1})
        double G, x;
        {
          const double qo = shfl_xor_d(q, 32), zo = shfl_xor_d(z1, 32);
          const double qh = bot ? qo : q, qb = bot ? q : qo, zh = bot ? zo : z1, zb = bot ? z1 : zo;
          const double eh = S.p.e[NP / 2 - 1];
          G = rcp_acc(fmax(fma(-eh * qb, eh, rcp_acc(qh)), sp1));
          x = G * fma(-eh * qb, zb, zh);
          if (!bot) S.p.d[j] = G;
        }
#pragma unroll 1
        for (int t = NB / 2 - 1; t >= 0; --t) {
#pragma unroll
          for (int h = 1; h >= 0; --h) {
            asm volatile("" ::: "memory");
            double iv[8], zi[8], ev[8], tv[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const int k = 16 * t + 8 * h + i;
              iv[i] = aa[at(t, 8 * h + i)];
              zi[i] = gg[at(t, 8 * h + i)];
              ev[i] = ee[k];
              tv[i] = c1[k];
            }
#pragma unroll
            for (int i = 7; i >= 0; --i) {
              double r = -ev[i] * iv[i];
              const double gn = fma(r * r, G, iv[i]), xn = fma(r, x, zi[i]);
              if (h == 1 && i == 7) {
                // row h itself: G and x as they are, and 1 for tau
                const bool mid = !bot && t == NB / 2 - 1;
                G = mid ? G : gn;
                x = mid ? x : xn;
                r = mid ? 1.0 : r;
              } else {
                G = gn;
                x = xn;
              }
              aa[at(t, 8 * h + i)] = r;
              gg[at(t, 8 * h + i)] = G;
              tv[i] = DUAL ? wj * x : wj * fma(-s, x, tv[i]);
              if (tl) cc[16 * t + 8 * h + i] = x;
            }
            // sums over the poles: of each 32 lanes the lower 16 keep steps 0..3
            // of the eight, the upper 16 steps 4..7
            const bool up = (lane & 16) != 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const double give = up ? tv[i] : tv[i + 4], keep = up ? tv[i + 4] : tv[i];
              tv[i] = row_sum16(keep + shfl_xor_d(give, 16));
            }
            if (lc == 0) {
#pragma unroll
              for (int i = 0; i < 4; ++i) c1[16 * t + 8 * h + (up ? 4 : 0) + i] = tv[i];
            }
          }
        }
      }
    } else if (batch == 0) {
      // ---- T_b of the reflector blocks ----
      for (int b = wave - 1; b < nblk; b += NB - 1) {
        const int k = 16 * b + lc;
        const double* src = V + (size_t)k * NP;
        d4 g = {0.0, 0.0, 0.0, 0.0};
        for (int k0 = 4 * b; k0 < 4 * nt; k0 += 4) {
          double xv[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) xv[u] = src[4 * (k0 + u) + lr];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const double xm = (k < n - 2 && 4 * (k0 + u) + lr > k) ? xv[u] : 0.0;
            g = mfma_f64(xm, xm, g);
          }
        }
        const double tk = src[k];
        const double tau = k < n - 2 ? tk : 0.0;
        // V^T V packed into the block's place, then column by column replaced:
        // T_b[j][j] = tau_j, T_b[0:j, j] = -tau_j T_b[0:j, 0:j] (V^T V)[0:j, j]
        double* gs = S.tp + b * 136;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (lr + 4 * r <= lc) gs[lc * (lc + 1) / 2 + lr + 4 * r] = g[r];
        __builtin_amdgcn_wave_barrier();
        double tr[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          asm volatile("" ::: "memory");  // column by column, not all loads at once
          double sm = 0.0;
#pragma unroll
          for (int q = 0; q < j; ++q) sm = fma(tr[q], gs[j * (j + 1) / 2 + q], sm);
          const double tj = readlane_d(tau, j);
          tr[j] = lane < j ? -tj * sm : (lane == j ? tj : 0.0);
          __builtin_amdgcn_wave_barrier();
          if (lane <= j) gs[j * (j + 1) / 2 + lane] = tr[j];
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
    lds_barrier();
    if (!DEEP && S.count != 1) return false;
    if (DEEP && S.count == 0) break;
    // F = T^-1/2: what the blocks before this one gave
    if (batch > 0) {
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) f[I][r] = Fz[(size_t)(16 * row_of(I) + lr + 4 * r) * NP + 16 * J + lc];
    } else {
#pragma unroll
      for (int I = 0; I < NB; ++I) f[I] = d4{0.0, 0.0, 0.0, 0.0};
    }
    // column lc of tile J from arr, times the weights of the lane's eight poles
    auto column_factors = [&](const double* arr, double (&o)[8]) {
      const int blk = S.first + batch;
      const int row = 16 * tile_of(J) + (low ? 15 - lc : lc);
      load_poles4(arr, row, 2 * lr, reinterpret_cast<double(&)[4]>(o[0]));
      load_poles4(arr, row, 2 * lr + 1, reinterpret_cast<double(&)[4]>(o[4]));
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        double w = ptab[blk * kPoleBlock + 32 + 8 * lr + q];
        if (DUAL) w = w / (1.0 + ptab[blk * kPoleBlock + 8 * lr + q]);
        o[q] *= w;
      }
    };
    d4 fd = {0.0, 0.0, 0.0, 0.0};  // the diagonal tile
    {
      // lane (lr, lc) runs column lc outwards from its diagonal entry for its
      // eight poles; the sums over the poles reach every lr, which keeps rows
      // lr + 4 r of that triangle (i: the rows in elimination order)
      double g[8];
      column_factors(S.p.g, g);
      d4 us;
      const int lcs = low ? 15 - lc : lc, lrs = low ? 3 - lr : lr;
#pragma unroll
      for (int i = 15; i >= 0; --i) {
        if (i % 4 == 3) asm volatile("" ::: "memory");  // the reads of four rows at a time
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          double r[4];
          load_poles4(S.p.a, 16 * tile_of(J) + i, 2 * lr + h, r);
#pragma unroll
          for (int q = 0; q < 4; ++q) g[4 * h + q] *= i < lcs ? r[q] : 1.0;
        }
        const double sm =
            sum_xor32(sum_xor16(((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7]))));
        if (i % 4 == 3) us[i / 4] = 0.0;
        us[i / 4] = (lrs == (i & 3) && i <= lcs) ? sm : us[i / 4];
      }
      // the other triangle: the transpose by a product with the identity (exact)
      d4 ut;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ut[r] = low ? us[3 - r] : us[r];
        fd[r] = 4 * r + lr == lc ? 0.0 : ut[r];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) fd = mfma_f64(ut[r], 4 * r + lr == lc ? 1.0 : 0.0, fd);
    }
    if (tid < NP) {
      const int k = step_row<NP>(tid);
      if (batch == 0) S.c[0][tid] = S.p.c[0][k];
      S.c[1][tid] = S.p.c[1][k] + (batch == 0 ? 0.0 : S.c[1][tid]);
    }
    lds_barrier();
    // towards the middle edge of a row's tile: alpha = tau_i ... (row i to the
    // edge), beta = G_ii times the tau between the outer edge and row i
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
    // off the diagonal: rows from arr, columns in B, both relative to the tile
    // edges (alpha of a tile's outermost row is the tile's whole product); four
    // poles at a time keep the operands few
    auto tile = [&](const double* arr, int I, double (&B)[8], d4 acc) {
      const int rI = row_of(I), t16 = 16 * tile_of(rI);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        double av[4], edge[4];
        load_poles4(arr, t16 + (rI < NB / 2 ? lc : 15 - lc), 2 * lr + h, av);
        load_poles4(S.p.a, t16, 2 * lr + h, edge);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          acc = mfma_f64(av[q], B[4 * h + q], acc);
          B[4 * h + q] *= edge[q];
        }
        asm volatile("" ::: "memory");
      }
      return acc;
    };
    {
      double B[8];
      column_factors(S.p.g, B);
#pragma unroll
      for (int I = NB / 2 - 2; I >= 0; --I)  // outside
        if (I < Js && J < nt && row_of(I) < nt) f[I] = tile(S.p.a, I, B, f[I]);
      column_factors(S.p.a, B);
#pragma unroll
      for (int I = 1; I < NB; ++I) {  // towards the middle, and beyond it
        if (I == NB / 2) {
#pragma unroll
          for (int q = 0; q < 8; ++q) B[q] *= S.p.d[8 * lr + q];
        }
        if (I > Js && J < nt && row_of(I) < nt) f[I] = tile(I < NB / 2 ? S.p.g : S.p.a, I, B, f[I]);
      }
#pragma unroll
      for (int I = 0; I < NB / 2; ++I)
        if (I == Js) f[I] += fd;
    }
    if (!DEEP || batch + 1 >= S.count) break;
    // another block: F so far to memory, d and Q^T 1 again
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) Fz[(size_t)(16 * row_of(I) + lr + 4 * r) * NP + 16 * J + lc] = f[I][r];
    lds_barrier();
    load_t();
    lds_barrier();
  }
  if (DEEP && S.count == 0) {
    // F, x and y from the eigenvectors, which go where M was
    const double bound = S.bound;
    if (tid < NP) {
      S.q.d[NP - 1 - tid] = dvec[(size_t)zl * NP + tid];
      S.q.e[tid] = tid < NP - 1 ? evec[(size_t)zl * NP + NP - 2 - tid] : 0.0;
      S.q.u[0][tid] = Vz[tid];
      S.q.u[1][tid] = Vz[2 * NP + tid];
    }
    __syncthreads();
    ql_functions<NP, 4 * NP, DUAL>(S.q, bound, Fz);
    if (tid < NP) {
      S.c[0][tid] = S.q.u[0][tid];
      S.c[1][tid] = S.q.u[1][tid];
    }
#pragma unroll
    for (int I = 0; I < NB; ++I) f[I] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int k = 0; k < NP; k += 4) {
      const double* zk = Fz + (size_t)(k + lr) * NP + lc;
      const double b = S.q.e[k + lr] * zk[16 * J];
#pragma unroll
      for (int I = 0; I < NB; ++I) f[I] = mfma_f64(zk[16 * row_of(I)], b, f[I]);
    }
  }
  // ---- R = Q F Q^T, [a, v] = Q [x, y] ----
  // thread t moves reflector pj of a block, rows pr + TPR e (loaded whole,
  // masked when stored: a load under a condition is waited for alone)
  double pf[ER];
  auto load_block = [&](int b, int pj, int pr) {
    const double* src = V + (size_t)(16 * b + pj) * NP + pr;
#pragma unroll
    for (int e = 0; e < ER; ++e) pf[e] = src[TPR * e];
  };
  load_block(nblk > 0 ? nblk - 1 : 0, tid / TPR, tid % TPR);
  lds_barrier();  // the pole arrays are read
#pragma unroll 1
  for (int b = nblk - 1; b >= 0; --b) {
    // the thread index made opaque in each pass: left visible, the addresses
    // and predicates made from it are computed ahead of the loop, and spill
    int tq = threadIdx.x;
    asm volatile("" : "+v"(tq));
    const int tid = tq, lr = (tq >> 4) & 3, lc = tq & 15, pj = tq / TPR, pr = tq % TPR;
    double* vb = S.m.vb[b & 1];
    const int k = 16 * b + pj;  // the reflector: zero up to row k (none past n - 3)
#pragma unroll
    for (int e = 0; e < ER; ++e) {
      const int r = pr + TPR * e;
      pf[e] = (k < n - 2 && r > k) ? pf[e] : 0.0;
      vb[r * LV + pj] = pf[e];
    }
    lds_barrier();
    double g0 = 0.0, g1 = 0.0;  // V^T [x, y]
#pragma unroll
    for (int e = 0; e < ER; ++e) {
      const int r = pr + TPR * e;
      g0 = fma(pf[e], S.c[0][r], g0);
      g1 = fma(pf[e], S.c[1][r], g1);
    }
    g0 = row_sum16(g0);
    g1 = row_sum16(g1);
    if (TPR == 32) {
      g0 = sum_xor16(g0);
      g1 = sum_xor16(g1);
    }
    if (pr == 0) {
      S.m.g[0][pj] = g0;
      S.m.g[1][pj] = g1;
    }
    // X^T = V^T F on the tile rows I >= b
    d4 y = {0.0, 0.0, 0.0, 0.0};
    {
      const double* vp = vb + lr * LV + lc;
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        asm volatile("" ::: "memory");  // the reads of later rows stay below
        const int rI = row_of(I);
        if (rI >= b && rI < nt && J < nt) {
          double va[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) va[q] = vp[(16 * rI + 4 * q) * LV];
#pragma unroll
          for (int q = 0; q < 4; ++q) y = mfma_f64(va[q], f[I][q], y);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) S.m.x[(16 * J + lc) * LV + lr + 4 * r] = y[r];
    __builtin_amdgcn_wave_barrier();
    {
      d4 sp = {0.0, 0.0, 0.0, 0.0};
      if (J >= b && J < nt) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int at = (16 * J + 4 * q + lr) * LV + lc;
          sp = mfma_f64(S.m.x[at], vb[at], sp);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (lr + 4 * r <= lc) S.m.s[wave][lc * (lc + 1) / 2 + lr + 4 * r] = sp[r];
    }
    const double* tp = S.tp + b * 136;
    // position of (lc, 4 q + lr) and its transpose in a packed triangle
    auto packed = [&](int q) {
      const int kk = 4 * q + lr, hi = kk > lc ? kk : lc, lo = kk > lc ? lc : kk;
      return hi * (hi + 1) / 2 + lo;
    };
    d4 pv = {0.0, 0.0, 0.0, 0.0};  // P
    if (J >= b && J < nt) {
      const double* vr = vb + (16 * J + lc) * LV + lr;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        pv = mfma_f64(4 * q + lr <= lc ? tp[packed(q)] : 0.0, vr[4 * q], pv);
    }
    lds_barrier();
    if (b > 0) load_block(b - 1, pj, pr);
    if (tid < 256) {  // S, T_b V^T [x, y]
      const int i = tid >> 4, hi = i > lc ? i : lc, lo = i > lc ? lc : i, at = hi * (hi + 1) / 2 + lo;
      double sm = S.m.s[0][at];
#pragma unroll
      for (int w = 1; w < NB; ++w) sm += S.m.s[w][at];
      S.m.sf[i * 17 + lc] = sm;
      const double tv = i <= lc ? tp[at] : 0.0;
      const double t0 = row_sum16(tv * S.m.g[0][lc]), t1 = row_sum16(tv * S.m.g[1][lc]);
      if (lc == 0) {
        S.m.t[0][i] = t0;
        S.m.t[1][i] = t1;
      }
    }
    lds_barrier();
    d4 qv = {0.0, 0.0, 0.0, 0.0};
    if (J >= b && J < nt) {
      d4 s2 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q) s2 = mfma_f64(S.m.sf[lc * 17 + 4 * q + lr], pv[q], s2);
#pragma unroll
      for (int q = 0; q < 4; ++q) y[q] -= s2[q];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) qv = mfma_f64(lc <= 4 * q + lr ? tp[packed(q)] : 0.0, y[q], qv);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      qv[q] = -qv[q];
      pv[q] = -pv[q];
    }
    if (tid < 2 * NP) {  // [x, y] <- [x, y] - V (T_b V^T [x, y])
      const int vq = tid / NP, r = tid % NP;
      const double2* v2 = reinterpret_cast<const double2*>(vb + r * LV);
      const double2* t2 = reinterpret_cast<const double2*>(S.m.t[vq]);
      double s0 = S.c[vq][r], s1 = 0.0;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const double2 vv = v2[c], tv = t2[c];
        s0 = fma(-vv.x, tv.x, s0);
        s1 = fma(-vv.y, tv.y, s1);
      }
      S.c[vq][r] = s0 + s1;
    }
    // F <- F - V qv - X pv, the second term for the tile columns J >= b (two
    // conditions without an else: with one, the tiles of both branches stay
    // live and spill)
    {
      const double* vp = vb + lc * LV + lr;
      const double* xp = S.m.x + lc * LV + lr;
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        asm volatile("" ::: "memory");  // the reads of later rows stay below
        const int rI = row_of(I);
        if (rI >= b && rI < nt && J < nt) {
          double vv[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) vv[q] = vp[16 * rI * LV + 4 * q];
#pragma unroll
          for (int q = 0; q < 4; ++q) f[I] = mfma_f64(vv[q], qv[q], f[I]);
        }
      }
      if (J >= b && J < nt) {
#pragma unroll
        for (int I = 0; I < NB; ++I) {
          asm volatile("" ::: "memory");
          double xv[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) xv[q] = xp[16 * row_of(I) * LV + 4 * q];
          if (row_of(I) < nt)
#pragma unroll
            for (int q = 0; q < 4; ++q) f[I] = mfma_f64(xv[q], pv[q], f[I]);
        }
      }
    }
  }
  TR* R = reinterpret_cast<TR*>(V);  // every reflector was read before the last barrier
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      R[(size_t)(16 * row_of(I) + lr + 4 * r) * NP + 16 * J + lc] = (TR)f[I][r];
  if (!DUAL && NP == 128) {  // R 1 (k_update128)
    double rs = 0.0;
#pragma unroll
    for (int I = 0; I < NB; ++I) rs += (f[I][0] + f[I][1]) + (f[I][2] + f[I][3]);
    rs = sum_xor32(sum_xor16(rs));
    if (lr == 0) Vz[16 * J + lc] = rs;
  }
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
    // R v = 1 / |M^1/2 1|
    if (!DUAL && NP == 128) Vz[3 * NP + tid] = tid < N ? 1.0 / sqrt(nv) : 0.0;
    if (ampl && tid < N) ampl[(size_t)z * N + tid] = ar;
    if (ar != ar) atomicOr(err, OAKG_DERR_NAN);
  }
  return true;
}

// The workgroup's LDS: one variable for k_func and for deep_zone, which it calls.
template <int NP>
__device__ __forceinline__ FuncLds<NP>& func_lds() {
  __shared__ FuncLds<NP> S;
  return S;
}

// A function of its own: inside k_func its loops made the tiles of every zone spill, and
// as kernels after k_func they cost 50 us of 1.2 ms at 5490 zones of N = 40 in waiting
// for a place on the device.
template <int NP, bool DUAL, typename TR>
__device__ __attribute__((noinline)) void deep_zone(int zl, int64_t z, int N, int64_t cnt,
                                                    const double* ptab, double* qmat, const double* dvec,
                                                    const double* evec, double* mat, double* vec,
                                                    double* ampl, unsigned* err) {
  func_zone<NP, DUAL, TR, true>(func_lds<NP>(), zl, z, N, cnt, ptab, qmat, dvec, evec, mat, vec, ampl,
                                      err);
}

template <int NP, bool DUAL, typename TR>
__global__ __launch_bounds__(4 * NP, 4) void k_func(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                    const int64_t* __restrict__ sel_ptr,
                                                    const double* __restrict__ ptab,
                                                    double* __restrict__ qmat,
                                                    const double* __restrict__ dvec,
                                                    const double* __restrict__ evec,
                                                    double* __restrict__ mat,
                                                    double* __restrict__ vec, double* __restrict__ ampl,
                                                    unsigned* __restrict__ err) {
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;  // the zone is solved by the other pipeline
  const int64_t cnt = sel_ptr[z + 1] - sel_ptr[z];
  if (cnt == 0) {  // no observations: a = 0
    if (threadIdx.x < NP) vec[(size_t)zl * 4 * NP + NP + threadIdx.x] = 0.0;
    return;
  }
  if (!func_zone<NP, DUAL, TR, false>(func_lds<NP>(), zl, z, N, cnt, ptab, qmat, dvec, evec, mat, vec,
                                            ampl, err)) {
    lds_barrier();
    deep_zone<NP, DUAL, TR>(zl, z, N, cnt, ptab, qmat, dvec, evec, mat, vec, ampl, err);
  }
}

// ===========================================================================
// N <= 32: the reduction, then R, a, v and the transform itself, a wave per
// zone (or for several) and no workgroup barrier
// ===========================================================================

template <typename F, int... K>
__device__ __forceinline__ void run_steps(F& f, std::integer_sequence<int, K...>) {
  (void)(f(std::integral_constant<int, K>()) && ...);
}

// The two 16-lane halves of each 32 lanes of v, each to both halves.
__device__ __forceinline__ void split16(double v, double& lo, double& hi) {
  const unsigned l = (unsigned)__double2loint(v), h = (unsigned)__double2hiint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(l, l, false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(h, h, false, false);
  lo = __hiloint2double((int)b[0], (int)a[0]);
  hi = __hiloint2double((int)b[1], (int)a[1]);
}

// M = Q T Q^T as launch_tridiag_lower64 leaves it (reflectors by rows with tau
// on the diagonal, rows N-2 and up not written; d, e; Q^T b, Q^T 1).  64 / NP
// zones share a wave: lane r of a zone holds row r of M in registers, the
// entries of v and w that the products need come from the other lanes by DPP
// row broadcasts, and the sums over rows by DPP, so that a step has neither an
// LDS access nor a barrier.  Bound by the issue of FP64 instructions: 16 N^2/2
// broadcasts and FMAs per zone and the four reductions of each step.  At N = 16
// 4096 zones take 10 us, 16384 zones 15 us (the reduction with the row vectors
// in LDS: 36 and 70 us).
template <int NP>
__global__ __launch_bounds__(64, 3) void k_tridiag_small(int64_t z0, const int32_t* __restrict__ zorder,
                                                         int nzc, int N,
                                                         const int64_t* __restrict__ sel_ptr,
                                                         const double* __restrict__ mat,
                                                         double* __restrict__ qmat,
                                                         double* __restrict__ dvec,
                                                         double* __restrict__ evec,
                                                         double* __restrict__ vec) {
  static_assert(NP == 16 || NP == 32, "");
  const int lane = threadIdx.x, r = lane % NP;
  const int zw = blockIdx.x * (64 / NP) + lane / NP;
  const int zl = zw < nzc ? zw : nzc - 1;
  const int64_t z = zone_at(zorder, z0 + zl);
  const bool active = zw < nzc && z >= 0 && sel_ptr[z < 0 ? 1 : z + 1] > sel_ptr[z < 0 ? 1 : z];
  if (__ballot(active) == 0) return;
  double* V = qmat + (size_t)zl * NP * NP;
  double* Vz = vec + (size_t)zl * 4 * NP;
  double x[NP];
  {
    const double2* row = reinterpret_cast<const double2*>(mat + (size_t)zl * NP * NP + (size_t)r * NP);
#pragma unroll
    for (int c = 0; c < NP / 2; ++c) {
      const double2 t = row[c];
      x[2 * c] = t.x;
      x[2 * c + 1] = t.y;
    }
  }
  double u0 = Vz[r], u1 = r < N ? 1.0 : 0.0;
  auto zone_sum = [](double s) {
    s = row_sum16(s);
    return NP == 32 ? sum_xor16(s) : s;
  };
  // step k as a constant: every register index and broadcast lane is one
  auto step = [&](auto kc) -> bool {
    constexpr int k = decltype(kc)::value;
    if (k >= N - 2) return false;
    // H = I - tau v v^T with H x = beta e_1, x = M[k+1.., k] (as in wide256.hip)
    const double sg = zone_sum(r > k + 1 ? x[k] * x[k] : 0.0);
    double lo = x[k], hi = x[k];
    if (NP == 32) split16(x[k], lo, hi);
    const double alpha = row_bcast(k + 1 < 16 ? lo : hi, k + 1);
    double tau = 0.0, scal = 0.0, beta = alpha;
    if (sg > 0x1p-900) {  // below: entries under 2^-450 of an M >= I, no reflection
      const double hh = fma(alpha, alpha, sg), aa = fabs(alpha);
      const double rn = rsqrt_acc(hh), nrm = hh * rn;
      beta = alpha >= 0.0 ? -nrm : nrm;
      tau = fma(aa, rn, 1.0);
      const double rd = rcp_acc(aa + nrm);
      scal = alpha >= 0.0 ? rd : -rd;
    }
    const double v = r > k + 1 ? x[k] * scal : (r == k + 1 ? 1.0 : 0.0);
    if (active) V[k * NP + r] = r == k ? tau : v;
    lo = hi = v;
    if (NP == 32) split16(v, lo, hi);
    double p0 = 0.0, p1 = 0.0;
#pragma unroll
    for (int c = k + 1; c < NP; ++c) {
      const double vc = row_bcast(c < 16 ? lo : hi, c);
      if (c & 1)
        p1 = fma(vc, x[c], p1);
      else
        p0 = fma(vc, x[c], p0);
    }
    const double p = p0 + p1;
    const double pv = zone_sum(v * p), s0 = zone_sum(v * u0), s1 = zone_sum(v * u1);
    const double w = r > k ? fma(-0.5 * tau * tau * pv, v, tau * p) : 0.0;
    u0 = fma(-tau * s0, v, u0);
    u1 = fma(-tau * s1, v, u1);
    x[k + 1] = r == k ? beta : x[k + 1];
    double wlo = w, whi = w;
    if (NP == 32) split16(w, wlo, whi);
#pragma unroll
    for (int c = k + 1; c < NP; ++c) {
      const double vc = row_bcast(c < 16 ? lo : hi, c), wc = row_bcast(c < 16 ? wlo : whi, c);
      x[c] = fma(-v, wc, fma(-w, vc, x[c]));
    }
    return true;
  };
  run_steps(step, std::make_integer_sequence<int, NP - 2>());
  // the diagonals: lane r's x[r] and x[r + 1]
  double d = x[0], e = x[1];
#pragma unroll
  for (int c = 1; c < NP; ++c) {
    d = r == c ? x[c] : d;
    if (c + 1 < NP) e = r == c ? x[c + 1] : e;
  }
  if (active) {
    dvec[(size_t)zl * NP + r] = d;
    if (r < NP - 1) evec[(size_t)zl * NP + r] = e;
    Vz[r] = u0;
    Vz[2 * NP + r] = u1;
  }
}

// R, a, v as k_func, and T = R Omega (analysis.hip) in place of M, for a zone
// per wave.  NP = 32: the two tiles on the diagonal are the halves of the
// elimination; NP = 16: one tile holds both halves.  In either case the
// entries that couple the halves are F_ik = sum_j w_j G_hh alpha_i alpha_k
// (alpha_i the product of the tau from row i to the middle).  With a wave
// holding the whole of F, X^T = V^T F is at once, in the accumulator layout,
// the A operand of X, and S that of S, so that only one transpose of X goes
// through the LDS.
// Bound by the chain of its phases at few zones (10 us for 64 zones of N = 16),
// by FP64 issue and the MFMAs (28 of 64 cycles per zone at NP = 16, 132 at
// NP = 32, for R) at many: 17 us for 4096 zones, 30 us for 16384.  QL sweeps,
// rotations, epilogue and k_tmat took 118 and 160 us.
template <int NP>
struct FuncSmallLds {
  static constexpr int NB = NP / 16;
  union {
    struct {
      double a[NP * 32];  // tau, then alpha
      double g[NP * 32];  // G_ii
      double d[NP], e[NP], c[2][NP];
    } p;
    struct {
      double x[NP * 18];
      double t[NB][16 * 17];  // V^T V, then T_b
      double v[NP];
    } m;
    struct {
      QlLds<NP> q;
      double z[NP * NP];  // its eigenvectors
    };
  };
};

template <int NP>
__global__ __launch_bounds__(64, NP == 16 ? 3 : 2) void k_func_small(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                      const int64_t* __restrict__ sel_ptr,
                                                      const double* __restrict__ ptab,
                                                      const double* __restrict__ qmat,
                                                      const double* __restrict__ dvec,
                                                      const double* __restrict__ evec,
                                                      double* __restrict__ mat, double* __restrict__ vec,
                                                      double* __restrict__ ampl, unsigned* __restrict__ err) {
  using L = FuncSmallLds<NP>;
  constexpr int NB = L::NB, H = NP / 2;
  __shared__ L S;
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;
  const int lane = threadIdx.x, lr = lane >> 4, lc = lane & 15;
  double* Vz = vec + (size_t)zl * 4 * NP;
  double* M = mat + (size_t)zl * NP * NP;
  if (sel_ptr[z + 1] == sel_ptr[z]) {  // no observations: T = I, a = 0
    if (lane < NP) Vz[NP + lane] = 0.0;
    for (int e = lane; e < NP * NP; e += 64) M[e] = (e / NP == e % NP) ? 1.0 : 0.0;
    return;
  }
  const double* V = qmat + (size_t)zl * NP * NP;
  const double dl = lane < NP ? dvec[(size_t)zl * NP + lane] : 0.0;
  const double u0 = lane < NP ? Vz[lane] : 0.0, u1 = lane < NP ? Vz[2 * NP + lane] : 0.0;
  if (lane < NP) {
    const int k = step_row<NP>(lane);
    S.p.d[k] = dl;
    S.p.e[k] = evec[(size_t)zl * NP + (lane < H ? lane : lane - 1)];
    S.p.c[0][k] = u0;
    S.p.c[1][k] = u1;
  }
  // reflector 16 b + lc, rows 4 q + lr (zero up to row k, none past N - 3)
  double va[NB][NP / 4], tau[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const double* src = V + (size_t)(16 * b + lc) * NP;
    tau[b] = src[16 * b + lc];
#pragma unroll
    for (int q = 0; q < NP / 4; ++q) va[b][q] = src[4 * q + lr];
  }
  lds_fence();
  // ---- pivots and solves: lanes 0..31 rows 0 .. H-1 downwards, one pole
  // each, lanes 32..63 the rest upwards ----
  double nt = 0.0;  // Gershgorin bound of T
  if (lane < NP)
    nt = fabs(S.p.d[lane]) + fabs(S.p.e[lane]) + (lane % H ? fabs(S.p.e[lane - 1]) : 0.0);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) nt = fmax(nt, shfl_xor_d(nt, o));
  const int ex = __builtin_amdgcn_readfirstlane(exponent_above(nt));
  const PoleBlocks pb = pole_blocks(ex > 1024 ? 0 : ex);  // infinities end as NaN in a
  d4 c[NB], f[NB][NB];
  if (pb.count > 0) {
#pragma unroll 1
    for (int batch = 0;; ++batch) {
      // the thread index made opaque in each pass (as in k_func)
      int lq = threadIdx.x;
      asm volatile("" : "+v"(lq));
      const int lane = lq, lr = lq >> 4, lc = lq & 15;
      const int j = lane & 31;
      const bool bot = lane >= 32;
      const int h0 = bot ? H : 0;
      double* aa = S.p.a + h0 * 32;
      double* gg = S.p.g + h0 * 32;
      const int jx = (j & ~1) ^ (H == 8 && bot ? 16 : 0);
      auto at = [&](int i) { return i * 32 + (jx ^ (2 * i)) + (j & 1); };
      double alpha[H], gh;  // alpha of the lane's rows and pole; G_hh
      const int blk = pb.first + batch;
      const bool tl = j == 31 && batch == 0;  // the lane of T itself
      {
        const double s = ptab[blk * kPoleBlock + j], sp1 = 1.0 + s, wj = ptab[blk * kPoleBlock + 32 + j];
        double* cc = S.p.c[tl ? 0 : 1] + h0;  // the lane's right-hand side
        double* c1 = S.p.c[1] + h0;
        double qv[H], zv[H], ev[H];
        double q = 0.0, z1 = 0.0, t = 0.0, e2 = 0.0;
#pragma unroll
        for (int i = 0; i < H; ++i) {
          ev[i] = S.p.e[h0 + i];
          q = rcp_acc(fmax(fma(-e2, q, S.p.d[h0 + i] + s), sp1));
          z1 = fma(t, z1, cc[i]);
          qv[i] = q;
          zv[i] = z1 * q;
          t = -ev[i] * q;
          e2 = ev[i] * ev[i];
        }
        const double qo = shfl_xor_d(q, 32), zo = shfl_xor_d(z1, 32);
        const double qh = bot ? qo : q, qb = bot ? q : qo, zh = bot ? zo : z1, zb = bot ? z1 : zo;
        const double eh = S.p.e[H - 1];
        double G = rcp_acc(fmax(fma(-eh * qb, eh, rcp_acc(qh)), sp1));
        double x = G * fma(-eh * qb, zb, zh), al = 1.0;
        gh = G;
        double tv[H];
#pragma unroll
        for (int i = H - 1; i >= 0; --i) {
          double rr = -ev[i] * qv[i];
          const double gn = fma(rr * rr, G, qv[i]), xn = fma(rr, x, zv[i]);
          const bool mid = i == H - 1 && !bot;  // row h itself
          G = mid ? G : gn;
          x = mid ? x : xn;
          rr = mid ? 1.0 : rr;
          al *= rr;
          alpha[i] = al;
          aa[at(i)] = rr;
          gg[at(i)] = G;
          tv[i] = wj * fma(-s, x, c1[i]);
          if (tl) cc[i] = x;
        }
        // sums over the poles: of each 32 lanes the lower 16 keep the first half
        // of the rows, the upper 16 the second
        const bool up = (lane & 16) != 0;
#pragma unroll
        for (int i = 0; i < H / 2; ++i) {
          const double give = up ? tv[i] : tv[i + H / 2], keep = up ? tv[i + H / 2] : tv[i];
          tv[i] = row_sum16(keep + shfl_xor_d(give, 16));
        }
        if (lc == 0) {
#pragma unroll
          for (int i = 0; i < H / 2; ++i) c1[(up ? H / 2 : 0) + i] = tv[i];
        }
      }
      lds_fence();
      // [x, y] as columns 0 and 1 of a tile per 16 rows
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double t = S.p.c[lc & 1][step_row<NP>(16 * I + lr + 4 * r)];
          c[I][r] = lc < 2 ? t : 0.0;
        }
      // ---- F = T^-1/2: each half's triangle outwards from its diagonal entries,
      // eight poles a lane, the other one by a product with the identity ----
      double w8[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) w8[q] = ptab[blk * kPoleBlock + 32 + 8 * lr + q];
#pragma unroll
      for (int J = 0; J < NB; ++J) {
        // column 16 J + lc is row lcs (elimination order) of half hb
        const bool hb = NP == 32 ? J == 1 : lc >= 8;
        const int lcs = hb ? 15 - lc : lc, base = NP == 32 ? 16 * J : (hb ? 8 : 0);
        double g[8];
        load_poles4(S.p.g, base + lcs, 2 * lr, reinterpret_cast<double(&)[4]>(g[0]));
        load_poles4(S.p.g, base + lcs, 2 * lr + 1, reinterpret_cast<double(&)[4]>(g[4]));
#pragma unroll
        for (int q = 0; q < 8; ++q) g[q] *= w8[q];
        const int lrs = hb ? 3 - lr : lr;
        d4 us = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = H - 1; i >= 0; --i) {
          if (i % 4 == 3) asm volatile("" ::: "memory");  // the reads of four rows at a time
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            double rr[4];
            load_poles4(S.p.a, base + i, 2 * lr + h, rr);
#pragma unroll
            for (int q = 0; q < 4; ++q) g[4 * h + q] *= i < lcs ? rr[q] : 1.0;
          }
          const double sm =
              sum_xor32(sum_xor16(((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7]))));
          us[i / 4] = (lrs == (i & 3) && i <= lcs) ? sm : us[i / 4];
        }
        d4 ut, fd;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          ut[r] = hb ? us[3 - r] : us[r];
          fd[r] = 4 * r + lr == lc ? 0.0 : ut[r];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) fd = mfma_f64(ut[r], 4 * r + lr == lc ? 1.0 : 0.0, fd);
        f[J][J] = fd;
      }
      // the entries between the halves
      lds_fence();
#pragma unroll
      for (int i = 0; i < H; ++i) aa[at(i)] = alpha[i];
      // G_hh of the poles 8 lr + q (lanes 0..31 hold them)
      double w8g[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) w8g[q] = w8[q] * shfl_d(gh, 8 * lr + q);
      lds_fence();
      {
        double av[NB][8];
#pragma unroll
        for (int I = 0; I < NB; ++I) {
          const int row = step_row<NP>(16 * I + lc);
          load_poles4(S.p.a, row, 2 * lr, reinterpret_cast<double(&)[4]>(av[I][0]));
          load_poles4(S.p.a, row, 2 * lr + 1, reinterpret_cast<double(&)[4]>(av[I][4]));
        }
        if (NP == 32) {
          f[0][NB - 1] = d4{0.0, 0.0, 0.0, 0.0};
          f[NB - 1][0] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            f[0][NB - 1] = mfma_f64(av[0][q], av[NB - 1][q] * w8g[q], f[0][NB - 1]);
            f[NB - 1][0] = mfma_f64(av[NB - 1][q], av[0][q] * w8g[q], f[NB - 1][0]);
          }
        } else {
          d4 x = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
          for (int q = 0; q < 8; ++q) x = mfma_f64(av[0][q], av[0][q] * w8g[q], x);
#pragma unroll
          for (int r = 0; r < 4; ++r) f[0][0][r] = (lc < 8) == (r < 2) ? f[0][0][r] : x[r];
        }
      }
      lds_fence();
      if (batch + 1 == pb.count) break;
      // another block: this one's F to memory (kept in registers it would cost the
      // zones of one block their occupancy), x and y to free slots, Q^T 1 again
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * I + lr + 4 * r;
#pragma unroll
          for (int J = 0; J < NB; ++J) M[row * NP + 16 * J + lc] = f[I][J][r];
          if (lc < 2) Vz[(lc ? 1 : 3) * NP + row] = c[I][r];
        }
      if (lane < NP) S.p.c[1][step_row<NP>(lane)] = Vz[2 * NP + lane];
      lds_fence();
    }
    if (pb.count == 2) {
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * I + lr + 4 * r;
#pragma unroll
          for (int J = 0; J < NB; ++J) f[I][J][r] += M[row * NP + 16 * J + lc];
          if (lc == 0) c[I][r] = Vz[3 * NP + row];
          if (lc == 1) c[I][r] += Vz[NP + row];
        }
    }
  } else {
    // from the eigenvectors
    if (lane < NP) {
      S.q.d[NP - 1 - lane] = dl;
      S.q.e[lane] = lane < NP - 1 ? evec[(size_t)zl * NP + NP - 2 - lane] : 0.0;
      S.q.u[0][lane] = u0;
      S.q.u[1][lane] = u1;
    }
    __syncthreads();
    ql_functions<NP, 64, false>(S.q, nt, S.z);
#pragma unroll
    for (int I = 0; I < NB; ++I) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double t = S.q.u[lc & 1][16 * I + lr + 4 * r];
        c[I][r] = lc < 2 ? t : 0.0;
      }
#pragma unroll
      for (int J = 0; J < NB; ++J) f[I][J] = d4{0.0, 0.0, 0.0, 0.0};
    }
#pragma unroll 1
    for (int k = 0; k < NP; k += 4) {
      const double* zk = S.z + (k + lr) * NP + lc;
#pragma unroll
      for (int J = 0; J < NB; ++J) {
        const double b = S.q.e[k + lr] * zk[16 * J];
#pragma unroll
        for (int I = 0; I < NB; ++I) f[I][J] = mfma_f64(zk[16 * I], b, f[I][J]);
      }
    }
    lds_fence();
  }
  // ---- T_b of the reflector blocks: lane i of row b of the wave has row i;
  // T_b[j][j] = tau_j, T_b[0:j, j] = -tau_j T_b[0:j, 0:j] (V^T V)[0:j, j] ----
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int k = 16 * b + lc;
#pragma unroll
    for (int q = 0; q < NP / 4; ++q) va[b][q] = (k < N - 2 && 4 * q + lr > k) ? va[b][q] : 0.0;
    tau[b] = k < N - 2 ? tau[b] : 0.0;
    d4 g = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 4 * b; q < NP / 4; ++q) g = mfma_f64(va[b][q], va[b][q], g);
#pragma unroll
    for (int r = 0; r < 4; ++r) S.m.t[b][(lr + 4 * r) * 17 + lc] = g[r];
  }
  lds_fence();
  {
    const int b = NB == 2 ? (lr & 1) : 0;
    const double tb = NB == 2 && b ? tau[NB - 1] : tau[0];
    double gr[16], sm[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      gr[q] = S.m.t[b][q * 17 + lc];
      sm[q] = 0.0;
    }
    lds_fence();
#pragma unroll
    for (int jj = 0; jj < 16; ++jj) {
      const double tj = row_bcast(tb, jj);
      const double tr = lc < jj ? -tj * sm[jj] : (lc == jj ? tj : 0.0);
      S.m.t[b][lc * 17 + jj] = tr;
#pragma unroll
      for (int q = jj + 1; q < 16; ++q) sm[q] = fma(row_bcast(gr[q], jj), tr, sm[q]);
    }
  }
  lds_fence();
  // ---- R = Q F Q^T, [a, v] = Q [x, y] ----
#pragma unroll
  for (int b = NB - 1; b >= 0; --b) {
    // V[16 I + lc][4 q + lr] of the block (the other operand form)
    double vt[NB][4], tA[4], tB[4];
#pragma unroll
    for (int I = b; I < NB; ++I)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int k = 16 * b + 4 * q + lr;
        const double t = V[(size_t)k * NP + 16 * I + lc];
        vt[I][q] = (k < N - 2 && 16 * I + lc > k) ? t : 0.0;
      }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      tA[q] = S.m.t[b][(4 * q + lr) * 17 + lc];
      tB[q] = S.m.t[b][lc * 17 + 4 * q + lr];
    }
    d4 y[NB], x[NB], pv[NB];
#pragma unroll
    for (int J = 0; J < NB; ++J) {
      y[J] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int I = b; I < NB; ++I)
#pragma unroll
        for (int q = 0; q < 4; ++q) y[J] = mfma_f64(va[b][4 * I + q], f[I][J][q], y[J]);
      x[J] = y[J];  // as an A operand: X, rows of tile J
      if (J >= b) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S.m.x[(16 * J + lc) * 18 + lr + 4 * r] = y[J][r];
      }
    }
    lds_fence();
    d4 s = {0.0, 0.0, 0.0, 0.0};  // S = X^T V
    d4 zc = {0.0, 0.0, 0.0, 0.0}, z2 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int J = b; J < NB; ++J)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        s = mfma_f64(S.m.x[(16 * J + 4 * q + lr) * 18 + lc], va[b][4 * J + q], s);
        zc = mfma_f64(va[b][4 * J + q], c[J][q], zc);
      }
#pragma unroll
    for (int q = 0; q < 4; ++q) z2 = mfma_f64(tB[q], zc[q], z2);
#pragma unroll
    for (int q = 0; q < 4; ++q) z2[q] = -z2[q];
#pragma unroll
    for (int J = b; J < NB; ++J) {
      pv[J] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        pv[J] = mfma_f64(tA[q], vt[J][q], pv[J]);
        c[J] = mfma_f64(vt[J][q], z2[q], c[J]);
      }
    }
#pragma unroll
    for (int J = 0; J < NB; ++J) {
      if (J >= b) {
        d4 s2 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q) s2 = mfma_f64(s[q], pv[J][q], s2);
#pragma unroll
        for (int q = 0; q < 4; ++q) y[J][q] -= s2[q];
      }
      d4 qv = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < 4; ++q) qv = mfma_f64(tB[q], y[J][q], qv);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        qv[q] = -qv[q];
        if (J >= b) pv[J][q] = -pv[J][q];
      }
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (I >= b) f[I][J] = mfma_f64(vt[I][q], qv[q], f[I][J]);
          if (J >= b) f[I][J] = mfma_f64(x[I][q], pv[J][q], f[I][J]);
        }
    }
    lds_fence();
  }
  // ---- a, v, and T = R Omega (k_tmat's formula) ----
  double vr[NB][4], nv = 0.0;
  bool nan = false;
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const double ar = row_bcast(c[I][r], 0);
      const int row = 16 * I + lr + 4 * r;
      vr[I][r] = row_bcast(c[I][r], 1);
      nv = fma(vr[I][r], vr[I][r], nv);
      nan = nan || ar != ar;
      if (lc == 0) {
        Vz[NP + row] = ar;
        if (ampl && row < N) ampl[(size_t)z * N + row] = ar;
      }
    }
  if (__ballot(nan) != 0 && lane == 0) atomicOr(err, OAKG_DERR_NAN);
  nv = 1.0 / sqrt(sum_xor32(sum_xor16(nv)));
  double vs = 0.0;
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      vr[I][r] *= nv;
      if (lc == 0) S.m.v[16 * I + lr + 4 * r] = vr[I][r];
      vs += 16 * I + lr + 4 * r < N - 1 ? vr[I][r] : 0.0;
    }
  vs = sum_xor32(sum_xor16(vs));
  lds_fence();
  const double wN = 1.0 / sqrt((double)N);
  const double vN = S.m.v[N - 1], sgv = vN >= 0 ? 1.0 : -1.0;
  const double alv = -1.0 / (fabs(vN) + 1.0), alw = -1.0 / (wN + 1.0), vw = vs * wN;
  // U = R [v, w~, z_v]
  d4 B[NB], U[NB];
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * I + lr + 4 * r;
      const double zv = vr[I][r] + (row == N - 1 ? sgv : 0.0);
      const double wt = row < N - 1 ? wN : 0.0;
      B[I][r] = lc == 0 ? vr[I][r] : (lc == 1 ? wt : (lc == 2 ? zv : 0.0));
    }
#pragma unroll
  for (int I = 0; I < NB; ++I) {
    U[I] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int K = 0; K < NB; ++K)
#pragma unroll
      for (int q = 0; q < 4; ++q) U[I] = mfma_f64(f[K][I][q], B[K][q], U[I]);
  }
#pragma unroll
  for (int J = 0; J < NB; ++J) {
    const int s = 16 * J + lc;
    const double zw = wN + (s == N - 1 ? 1.0 : 0.0), vt = s < N - 1 ? S.m.v[s] : 0.0;
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double u1 = row_bcast(U[I][r], 0), u2 = row_bcast(U[I][r], 1), u3 = row_bcast(U[I][r], 2);
        double t = s == N - 1 ? 0.0 : f[I][J][r];
        if (s < N) t += u1 * wN + alw * u2 * zw + alv * u3 * vt + alv * alw * vw * u3 * zw;
        M[(size_t)(16 * I + lr + 4 * r) * NP + s] = t;
      }
  }
}

// ===========================================================================
// N > 128: a zone's F is 512 KB, so the steps of k_func are kernels of their
// own (the others are in wide256.hip).
// ===========================================================================

// Pivots and solves as in k_func (wave 0), T_b of the reflector blocks (waves
// 1 to 3), then a = Q x and v = Q y / |Q y|.  For the products that form F, per
// row (in elimination order) and pole: tau and G_ii (the tiles on the
// diagonal), and alpha and beta relative to the tile edges; `poles` has these
// four arrays, of one block of poles and then of the other (or the eigenvectors,
// ql_zone256), tblk, after T_b, the weights and G_hh of each block (or the
// eigenvectors' weights) and the number of blocks (PoleSet256).  The recurrence
// leaves 1/gamma and z/gamma of the way in where tau and G go on the way out.
template <int NP>
struct PoleLds {
  union {
    struct {
      double d[NP], e[NP], c[2][NP];  // c: Q^T b, Q^T 1, then x, y (elimination order)
      double v[2][NP];                // x, y; then a, v
    };
    QlLds<NP> q;
  };
  double bound;  // of T's spectrum
  int count;
  double tp[NP / 16 * 136];       // T_b, packed
  double g[2][16], t[2][16], red[4];
};

__device__ __forceinline__ PoleLds<256>& pole_lds() {
  __shared__ PoleLds<256> S;
  return S;
}

// QL for a zone beyond the poles (a function of its own as deep_zone): the
// eigenvectors to Z.
__device__ __attribute__((noinline)) void ql_zone256(const double* d, const double* e, const double* Vz,
                                                     double* Z) {
  constexpr int NP = 256;
  PoleLds<NP>& S = pole_lds();
  const int tid = threadIdx.x;
  S.q.d[NP - 1 - tid] = d[tid];
  S.q.e[tid] = tid < NP - 1 ? e[NP - 2 - tid] : 0.0;
  S.q.u[0][tid] = Vz[tid];
  S.q.u[1][tid] = Vz[2 * NP + tid];
  __syncthreads();
  ql_functions<NP, 256, false>(S.q, S.bound, Z);
}

__global__ __launch_bounds__(256, 2) void k_pole256(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                    const int64_t* __restrict__ sel_ptr,
                                                    const double* __restrict__ ptab,
                                                    const double* __restrict__ qmat,
                                                    const double* __restrict__ dvec,
                                                    const double* __restrict__ evec, double* poles,
                                                    double* __restrict__ tblk,
                                                    double* __restrict__ vec, double* __restrict__ ampl,
                                                    unsigned* __restrict__ err) {
  constexpr int NP = 256, H = NP / 2;
  PoleLds<NP>& S = pole_lds();
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane >> 4, lc = lane & 15;
  double* Vz = vec + (size_t)zl * 4 * NP;
  if (sel_ptr[z + 1] == sel_ptr[z]) {  // no observations: a = 0
    Vz[NP + tid] = 0.0;
    return;
  }
  const double* V = qmat + (size_t)zl * NP * NP;
  const int nblk = N > 2 ? (N + 13) >> 4 : 0;
  {
    const int k = step_row<NP>(tid);
    S.d[k] = dvec[(size_t)zl * NP + tid];
    S.e[k] = evec[(size_t)zl * NP + (tid < H ? tid : tid - 1)];
    S.c[0][k] = Vz[tid];
    S.c[1][k] = Vz[2 * NP + tid];
  }
  lds_barrier();
  double* tz = tblk + (size_t)zl * NP * NP;
  double* P0 = poles + (size_t)zl * NP * NP;
  if (wave == 0) {
    double nt = 0.0;  // Gershgorin bound of T
#pragma unroll
    for (int h = 0; h < NP / 64; ++h) {
      const int k = lane + 64 * h;
      nt = fmax(nt, fabs(S.d[k]) + fabs(S.e[k]) + (k % H ? fabs(S.e[k - 1]) : 0.0));
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) nt = fmax(nt, shfl_xor_d(nt, o));
    const int ex = __builtin_amdgcn_readfirstlane(exponent_above(nt));
    const PoleBlocks pb = pole_blocks(ex > 1024 ? 0 : ex);  // infinities end as NaN in a
    if (lane == 0) {
      S.bound = nt;
      S.count = pb.count;
      tz[PoleSet256::kCount] = (double)pb.count;
    }
    const int j = lane & 31;
    const bool bot = lane >= 32, up = (lane & 16) != 0;
    // block by block, the one with T itself last: y adds up in v
#pragma unroll 1
    for (int batch = pb.count - 1; batch >= 0; --batch) {
      const int blk = pb.first + batch;
      const bool tl = j == 31 && batch == 0;  // the lane of T itself
      const double s = ptab[blk * kPoleBlock + j], sp1 = 1.0 + s, wj = ptab[blk * kPoleBlock + 32 + j];
      const int h0 = bot ? H : 0;
      const double* dd = S.d + h0;
      const double* ee = S.e + h0;
      double* cc = S.c[tl ? 0 : 1] + h0;  // the lane's right-hand side
      double* c1 = S.c[1] + h0;
      double* P = P0 + batch * PoleSet256::kArrays;
      double* pa = P + h0 * 32 + j;  // tau (first 1/gamma); + NP 32: G_ii (first z/gamma)
      double* pg = pa + NP * 32;
      double q = 0.0, z1 = 0.0, tau = 0.0, e2 = 0.0;
#pragma unroll 1
      for (int t = 0; t < H; t += 8) {
        double dv[8], ev[8], cv[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          dv[i] = dd[t + i];
          ev[i] = ee[t + i];
          cv[i] = cc[t + i];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          q = rcp_acc(fmax(fma(-e2, q, dv[i] + s), sp1));
          z1 = fma(tau, z1, cv[i]);
          pa[(t + i) * 32] = q;
          pg[(t + i) * 32] = z1 * q;
          tau = -ev[i] * q;
          e2 = ev[i] * ev[i];
        }
      }
      double G, x;
      {
        const double qo = shfl_xor_d(q, 32), zo = shfl_xor_d(z1, 32);
        const double qh = bot ? qo : q, qb = bot ? q : qo, zh = bot ? zo : z1, zb = bot ? z1 : zo;
        const double eh = S.e[H - 1];
        G = rcp_acc(fmax(fma(-eh * qb, eh, rcp_acc(qh)), sp1));
        x = G * fma(-eh * qb, zb, zh);
        if (!bot) {
          tz[PoleSet256::kWeights + 64 * batch + j] = wj;
          tz[PoleSet256::kWeights + 64 * batch + 32 + j] = G;
        }
      }
#pragma unroll 1
      for (int t = H - 16; t >= 0; t -= 16) {
        double r[16], g[16];  // 1/gamma and z/gamma, then tau and G_ii
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          r[i] = pa[(t + i) * 32];
          g[i] = pg[(t + i) * 32];
        }
#pragma unroll
        for (int h = 1; h >= 0; --h) {
          double tv[8];
#pragma unroll
          for (int i = 7; i >= 0; --i) {
            const int k = 8 * h + i;
            double rr = -ee[t + k] * r[k];
            const double gn = fma(rr * rr, G, r[k]), xn = fma(rr, x, g[k]);
            const bool mid = k == 15 && !bot && t == H - 16;  // row h itself
            G = mid ? G : gn;
            x = mid ? x : xn;
            rr = mid ? 1.0 : rr;
            r[k] = rr;
            g[k] = G;
            tv[i] = wj * fma(-s, x, c1[t + k]);
            if (tl) cc[t + k] = x;
          }
          // sums over the poles, as in k_func
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const double give = up ? tv[i] : tv[i + 4], keep = up ? tv[i + 4] : tv[i];
            tv[i] = row_sum16(keep + shfl_xor_d(give, 16));
          }
          if (lc == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) c1[t + 8 * h + (up ? 4 : 0) + i] = tv[i];
          }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          pa[(t + i) * 32] = r[i];
          pg[(t + i) * 32] = g[i];
        }
        // towards the middle edge of the tile: alpha, beta
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
          pa[2 * NP * 32 + (t + i) * 32] = r[i];
          pg[2 * NP * 32 + (t + i) * 32] = g[i];
        }
      }
      if (pb.count > 1) {
        // y of both blocks, Q^T 1 again in between
        lds_fence();
#pragma unroll
        for (int h = 0; h < NP / 64; ++h) {
          const int k = lane + 64 * h, r = step_row<NP>(k);
          if (batch > 0) {
            S.v[1][k] = S.c[1][k];
            S.c[1][k] = Vz[2 * NP + r];
          } else {
            S.c[1][k] += S.v[1][k];
          }
        }
        lds_fence();
      }
    }
  } else {
    for (int b = wave - 1; b < nblk; b += 3) {
      const int k = 16 * b + lc;
      // V^T V packed into the block's place, then column by column replaced
      d4 g = {0.0, 0.0, 0.0, 0.0};
      for (int k0 = 4 * b; k0 < NP / 4; k0 += 4) {
        double xv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) xv[u] = *reflector256(V, k, 4 * (k0 + u) + lr);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const double xm = (k < N - 2 && 4 * (k0 + u) + lr > k) ? xv[u] : 0.0;
          g = mfma_f64(xm, xm, g);
        }
      }
      const double tk = *reflector256(V, k, k);
      const double tau = k < N - 2 ? tk : 0.0;
      double* gs = S.tp + b * 136;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (lr + 4 * r <= lc) gs[lc * (lc + 1) / 2 + lr + 4 * r] = g[r];
      lds_fence();
      double tr[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        double sm = 0.0;
#pragma unroll
        for (int q = 0; q < j; ++q) sm = fma(tr[q], gs[j * (j + 1) / 2 + q], sm);
        const double tj = readlane_d(tau, j);
        tr[j] = lane < j ? -tj * sm : (lane == j ? tj : 0.0);
        lds_fence();
        if (lane <= j) gs[j * (j + 1) / 2 + lane] = tr[j];
      }
      lds_fence();
    }
  }
  lds_barrier();
  if (S.count == 0) {  // x and y where v is
    static_assert(offsetof(PoleLds<NP>, v) == offsetof(PoleLds<NP>, q) + offsetof(QlLds<NP>, u), "");
    ql_zone256(dvec + (size_t)zl * NP, evec + (size_t)zl * NP, Vz, P0);
    tz[PoleSet256::kWeights + tid] = S.q.e[tid];
  } else {
    const int k = step_row<NP>(tid);
    const double x = S.c[0][k], y = S.c[1][k];
    S.v[0][tid] = x;
    S.v[1][tid] = y;
  }
  for (int e = tid; e < nblk * 136; e += 256) tz[e] = S.tp[e];
  // [a, v] = Q [x, y]: thread (pj, pr) has rows pr + 16 e of reflector pj of a block
  const int pj = tid >> 4, pr = tid & 15;
  double pf[16];
  auto load_block = [&](int b) {
#pragma unroll
    for (int e = 0; e < 16; ++e) pf[e] = *reflector256(V, 16 * b + pj, pr + 16 * e);
  };
  if (nblk > 0) load_block(nblk - 1);
  lds_barrier();
#pragma unroll 1
  for (int b = nblk - 1; b >= 0; --b) {
    const int k = 16 * b + pj;
    double g0 = 0.0, g1 = 0.0;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      pf[e] = (k < N - 2 && pr + 16 * e > k) ? pf[e] : 0.0;
      g0 = fma(pf[e], S.v[0][pr + 16 * e], g0);
      g1 = fma(pf[e], S.v[1][pr + 16 * e], g1);
    }
    g0 = row_sum16(g0);
    g1 = row_sum16(g1);
    if (pr == 0) {
      S.g[0][pj] = g0;
      S.g[1][pj] = g1;
    }
    lds_barrier();
    // t = T_b g (row pj of T_b, column pr)
    const double tv = pj <= pr ? S.tp[b * 136 + pr * (pr + 1) / 2 + pj] : 0.0;
    const double t0 = row_sum16(tv * S.g[0][pr]), t1 = row_sum16(tv * S.g[1][pr]);
    if (pr == 0) {
      S.t[0][pj] = t0;
      S.t[1][pj] = t1;
    }
    lds_barrier();
    // thread r: row r of [x, y] less V t
    double s0 = S.v[0][tid], s1 = S.v[1][tid];
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const double vv = 16 * b + c < N - 2 && tid > 16 * b + c ? *reflector256(V, 16 * b + c, tid) : 0.0;
      s0 = fma(-vv, S.t[0][c], s0);
      s1 = fma(-vv, S.t[1][c], s1);
    }
    S.v[0][tid] = s0;
    S.v[1][tid] = s1;
    if (b > 0) load_block(b - 1);
    lds_barrier();
  }
  const double ar = S.v[0][tid], vr = S.v[1][tid];
  const double nv = wave_sum_fast(vr * vr);
  if (lane == 0) S.red[wave] = nv;
  lds_barrier();
  Vz[NP + tid] = ar;
  Vz[2 * NP + tid] = vr / sqrt((S.red[0] + S.red[1]) + (S.red[2] + S.red[3]));
  if (ampl && tid < N) ampl[(size_t)z * N + tid] = ar;
  if (ar != ar) atomicOr(err, OAKG_DERR_NAN);
}

// R = Y Y^T from the Y = U diag(mu^-1/4) of the Jacobi option, so that one form
// reaches the transform.
template <int NP, typename TR>
__global__ __launch_bounds__(256) void k_yyt(int64_t z0, const int32_t* __restrict__ zorder,
                                             const int64_t* __restrict__ sel_ptr,
                                             double* __restrict__ ymat) {
  constexpr int LD = NP + 1, NB = NP / 16;
  __shared__ double Y[NP * LD];
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;
  if (sel_ptr[z + 1] == sel_ptr[z]) return;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane >> 4, lc = lane & 15;
  double* Yz = ymat + (size_t)zl * NP * NP;
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
}

// R 1 and R v in slots 0 and 3 of vec, as k_func leaves them at NP = 128 (R is
// symmetric: a thread per column).
template <int NP, typename TR>
__global__ __launch_bounds__(NP) void k_row_sums(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                 const int64_t* __restrict__ sel_ptr,
                                                 const double* __restrict__ ymat, double* vec) {
  const int zl = blockIdx.x, c = threadIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0 || sel_ptr[z + 1] == sel_ptr[z]) return;
  const TR* R = reinterpret_cast<const TR*>(ymat + (size_t)zl * NP * NP);
  double* Vz = vec + (size_t)zl * 4 * NP;
  double s1 = 0.0, sv = 0.0;
  for (int s = 0; s < N; ++s) {
    const double x = (double)R[(size_t)s * NP + c];
    s1 += x;
    sv = fma(x, Vz[2 * NP + s], sv);
  }
  Vz[c] = s1;
  Vz[3 * NP + c] = sv;
}

// What Omega adds to the rows of R (OmegaRow), from R 1, R v and row N - 1 of R: p
// and q in place of the first two, row N - 1 of (R Omega)^T in that of the last.
template <int NP, typename TR>
__global__ __launch_bounds__(NP) void k_omega_rows(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                   const int64_t* __restrict__ sel_ptr, double* ymat,
                                                   double* vec) {
  __shared__ double red[NP / 64];
  const int zl = blockIdx.x, c = threadIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0 || sel_ptr[z + 1] == sel_ptr[z]) return;
  TR* last = reinterpret_cast<TR*>(ymat + (size_t)zl * NP * NP) + (size_t)(N - 1) * NP + c;
  double* Vz = vec + (size_t)zl * 4 * NP;
  const double r1 = Vz[c], kv = Vz[3 * NP + c], rN = (double)*last, vN = Vz[2 * NP + N - 1];
  const double s = wave_sum_fast(c < N - 1 ? Vz[2 * NP + c] : 0.0);
  if ((c & 63) == 0) red[c >> 6] = s;
  __syncthreads();
  double sv = 0.0;
#pragma unroll
  for (int w = 0; w < NP / 64; ++w) sv += red[w];
  const OmegaRow o = omega_row(N, kv, r1, rN, vN, sv);
  Vz[c] = o.p;
  Vz[3 * NP + c] = o.q;
  *last = (TR)(o.p + o.l);
}

void launch_omega_rows128(const ChunkArgs& A, hipStream_t st) {
  if (A.prec == 1)
    hipLaunchKernelGGL((k_omega_rows<128, float>), dim3(A.nzc), dim3(128), 0, st, A.z0, A.zorder, A.N,
                       A.sel_ptr, A.ymat, A.vec);
  else
    hipLaunchKernelGGL((k_omega_rows<128, double>), dim3(A.nzc), dim3(128), 0, st, A.z0, A.zorder, A.N,
                       A.sel_ptr, A.ymat, A.vec);
}

// The reduction (wide256.hip) and the functions of T for a chunk at NP = 64
// or 128 (dual: the observation-space zones).
void launch_func(int NP, const ChunkArgs& A, bool dual, hipStream_t st) {
#define OAK_FUNC(P, D, TR)                                                                     \
  hipLaunchKernelGGL((k_func<P, D, TR>), dim3(A.nzc), dim3(4 * P), 0, st, A.z0, A.zorder, A.N, \
                     A.sel_ptr, A.poles, A.ymat, A.dvec, A.evec, A.mat, A.vec, A.ampl, A.err)
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

// NP = 16, 32: M and b of a chunk to T = R Omega (in place of M), a and v.
void launch_func_small(int NP, const ChunkArgs& A, hipStream_t st) {
#define OAK_SMALL(P)                                                                               \
  do {                                                                                             \
    hipLaunchKernelGGL(k_tridiag_small<P>, dim3((A.nzc + 64 / P - 1) / (64 / P)), dim3(64), 0, st, \
                       A.z0, A.zorder, A.nzc, A.N, A.sel_ptr, A.mat, A.ymat, A.dvec, A.evec,       \
                       A.vec);                                                                     \
    hipLaunchKernelGGL(k_func_small<P>, dim3(A.nzc), dim3(64), 0, st, A.z0, A.zorder, A.N,         \
                       A.sel_ptr, A.poles, A.ymat, A.dvec, A.evec, A.mat, A.vec, A.ampl, A.err);            \
  } while (0)
  if (NP == 16)
    OAK_SMALL(16);
  else
    OAK_SMALL(32);
#undef OAK_SMALL
}

// N > 128: the pole arrays to umat, T_b (and the weights) to the rows of ymat that the reduction's
// trailing block leaves (128 .. 191), a and v.
void launch_pole256(const ChunkArgs& A, hipStream_t st) {
  hipLaunchKernelGGL(k_pole256, dim3(A.nzc), dim3(256), 0, st, A.z0, A.zorder, A.N, A.sel_ptr, A.poles,
                     A.ymat, A.dvec, A.evec, A.umat, A.ymat + 128 * 256, A.vec, A.ampl, A.err);
}

void launch_yyt(int NP, const ChunkArgs& A, hipStream_t st) {
  const dim3 g(A.nzc), b(256);
#define OAK_YYT(P, TR) \
  hipLaunchKernelGGL((k_yyt<P, TR>), g, b, 0, st, A.z0, A.zorder, A.sel_ptr, A.ymat)
  if (NP == 64)
    OAK_YYT(64, double);
  else if (A.prec == 1)
    OAK_YYT(128, float);
  else
    OAK_YYT(128, double);
#undef OAK_YYT
  if (NP == 64) return;
  if (A.prec == 1)
    hipLaunchKernelGGL((k_row_sums<128, float>), g, dim3(128), 0, st, A.z0, A.zorder, A.N, A.sel_ptr,
                       A.ymat, A.vec);
  else
    hipLaunchKernelGGL((k_row_sums<128, double>), g, dim3(128), 0, st, A.z0, A.zorder, A.N, A.sel_ptr,
                       A.ymat, A.vec);
}

}  // namespace oakg
