// Householder reduction of a symmetric matrix of up to 64 rows on one wave: the
// N = 33..64 eigensolve, the observation-space zones of N = 128, and the trailing
// 64 x 64 block that k_tridiag_lower leaves of a larger matrix.
#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"

namespace oakg {

namespace {

// acc += A v over the eight columns of one column block: entry c of v, in lane
// c % 16 of every row of 16 lanes of vb, multiplies the lane's own a[c].  The
// broadcast is part of the multiply-add (DPP row_newbcast, which the compiler
// leaves as a move of its own); two wait states lie between a VALU write of vb
// and the first of them.
#define OAK_DPP(C) " row_newbcast:" #C " row_mask:0xf bank_mask:0xf\n\t"
#define OAK_MV8(C0, C1, C2, C3, C4, C5, C6, C7)                                             \
  asm("s_nop 1\n\t"                                                                         \
      "v_fmac_f64_dpp %0, %4, %5" OAK_DPP(C0) "v_fmac_f64_dpp %1, %4, %6" OAK_DPP(C1)        \
      "v_fmac_f64_dpp %2, %4, %7" OAK_DPP(C2) "v_fmac_f64_dpp %3, %4, %8" OAK_DPP(C3)        \
      "v_fmac_f64_dpp %0, %4, %9" OAK_DPP(C4) "v_fmac_f64_dpp %1, %4, %10" OAK_DPP(C5)       \
      "v_fmac_f64_dpp %2, %4, %11" OAK_DPP(C6) "v_fmac_f64_dpp %3, %4, %12" OAK_DPP(C7)      \
      : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3])                                      \
      : "v"(vb), "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), \
        "v"(a[7]))
// a[c] += xb_c y for the eight columns
#define OAK_UP8(C0, C1, C2, C3, C4, C5, C6, C7)                                             \
  asm("s_nop 1\n\t"                                                                         \
      "v_fmac_f64_dpp %0, %8, %9" OAK_DPP(C0) "v_fmac_f64_dpp %1, %8, %9" OAK_DPP(C1)        \
      "v_fmac_f64_dpp %2, %8, %9" OAK_DPP(C2) "v_fmac_f64_dpp %3, %8, %9" OAK_DPP(C3)        \
      "v_fmac_f64_dpp %4, %8, %9" OAK_DPP(C4) "v_fmac_f64_dpp %5, %8, %9" OAK_DPP(C5)        \
      "v_fmac_f64_dpp %6, %8, %9" OAK_DPP(C6) "v_fmac_f64_dpp %7, %8, %9" OAK_DPP(C7)        \
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]),  \
        "+v"(a[7])                                                                          \
      : "v"(xb), "v"(y))

// HALF: the column block is the upper half of its 16 columns
template <int HALF>
__device__ __forceinline__ void row_dot8(double (&s)[4], double vb, const double* a) {
  if constexpr (HALF)
    OAK_MV8(8, 9, 10, 11, 12, 13, 14, 15);
  else
    OAK_MV8(0, 1, 2, 3, 4, 5, 6, 7);
}
template <int HALF>
__device__ __forceinline__ void row_add8(double* a, double xb, double y) {
  if constexpr (HALF)
    OAK_UP8(8, 9, 10, 11, 12, 13, 14, 15);
  else
    OAK_UP8(0, 1, 2, 3, 4, 5, 6, 7);
}
#undef OAK_UP8
#undef OAK_MV8
#undef OAK_DPP

struct Tri64 {
  double v[64], w[64];
};

// Steps 8 B .. 8 B + 7 (those below n - 2); a: the lane's row, x: column i
// from the diagonal on, u: entries of b and 1_N.
template <int B>
__device__ __forceinline__ void tri_steps(Tri64& S, double (&a)[64], double& x, double (&u)[2],
                                          bool has_u, int n, int lane, double* V, int ldv,
                                          double* dv, double* ev, int64_t dstep) {
  constexpr int C0 = 8 * B, Q0 = C0 / 16;
  const int end = n - 2 < C0 + 8 ? n - 2 : C0 + 8;
  for (int i = C0; i < end; ++i) {
    // reflector H = I - tau v v^T with H x = beta e_1, x = A[i+1.., i]; the
    // products with u over the rows that scal multiplies beside the norm
    const double xs = lane >= i + 2 ? x : 0.0;
    double s = xs * xs, su0 = xs * u[0], su1 = xs * u[1];
    s = wave_sum_d(s);
    su0 = wave_sum_d(su0);
    su1 = wave_sum_d(su1);
    const double alpha = readlane_d(x, i + 1), di = readlane_d(x, i);
    double tau = 0.0, scal = 0.0, beta = alpha;
    if (s > 0.0) {
      // beta = -sign(alpha) nrm, tau = (beta - alpha) / beta = 1 + |alpha| / nrm,
      // 1 / (alpha - beta) = sign(alpha) / (|alpha| + nrm)
      const double hh = fma(alpha, alpha, s);
      const double aa = fabs(alpha);
      if (hh > 0x1p-900 && hh < 0x1p+900) {
        const double rn = rsqrt_acc(hh);
        const double nrm = hh * rn;
        beta = alpha >= 0.0 ? -nrm : nrm;
        tau = fma(aa, rn, 1.0);
        const double rd = rcp_acc(aa + nrm);
        scal = alpha >= 0.0 ? rd : -rd;
      } else {
        const double nrm = sqrt(hh);
        beta = alpha >= 0.0 ? -nrm : nrm;
        tau = (beta - alpha) / beta;
        scal = 1.0 / (alpha - beta);
      }
    }
    const double v = lane == i + 1 ? 1.0 : xs * scal;
    S.v[lane] = v;
    lds_fence();
    double vb[4];
#pragma unroll
    for (int q = Q0; q < 4; ++q) vb[q] = S.v[16 * q + (lane & 15)];
    V[(size_t)i * ldv + lane] = lane == i ? tau : v;
    if (lane == 0) {
      dv[i * dstep] = di;
      ev[i * dstep] = beta;
    }
    if (has_u) {
      u[0] = fma(-tau * fma(scal, su0, readlane_d(u[0], i + 1)), v, u[0]);
      u[1] = fma(-tau * fma(scal, su1, readlane_d(u[1], i + 1)), v, u[1]);
    }
    // p = tau A v, w = p - (tau/2)(v^T p) v
    double ps[4] = {};
#pragma unroll
    for (int c = C0; c < 64; c += 16) {
      if ((c & 15) == 0) {
        row_dot8<0>(ps, vb[c / 16], a + c);
        row_dot8<1>(ps, vb[c / 16], a + c + 8);
      } else {
        row_dot8<1>(ps, vb[c / 16], a + c);
        if (c + 8 < 64) row_dot8<0>(ps, vb[(c + 8) / 16], a + c + 8);
      }
    }
    const double p = lane > i ? tau * ((ps[0] + ps[1]) + (ps[2] + ps[3])) : 0.0;
    const double K = -0.5 * tau * wave_sum_d(v * p);
    const double w = fma(K, v, p);
    S.w[lane] = w;
    lds_fence();
    double wb[4];
#pragma unroll
    for (int q = Q0; q < 4; ++q) wb[q] = S.w[16 * q + (lane & 15)];
    // A -= v w^T + w v^T
    const double nv = -v, nw = -w;
#pragma unroll
    for (int c = C0; c < 64; c += 8) {
      if ((c & 15) == 0) {
        row_add8<0>(a + c, vb[c / 16], nw);
        row_add8<0>(a + c, wb[c / 16], nv);
      } else {
        row_add8<1>(a + c, vb[c / 16], nw);
        row_add8<1>(a + c, wb[c / 16], nv);
      }
    }
    // column i + 1: entry i + 1 of the lane's row
    double nx = a[C0 + 1];
#pragma unroll
    for (int j = 2; j <= 8; ++j)
      if (C0 + j < 64) nx = i + 1 == C0 + j ? a[C0 + j < 64 ? C0 + j : 63] : nx;
    x = lane > i ? nx : 0.0;
  }
}

}  // namespace

// One wave per zone, lane r holding row r of the full matrix in registers: A v
// and the rank-2 update need no sums over lanes, v and w reach every lane as
// four values per row of 16 lanes (one write and four reads of LDS each) that the
// multiply-adds broadcast from, and the columns that are done drop out in eights.
// Bound by VALU issue: about 110 multiply-adds and as much again for the four
// sums over the wave, the reflector and the stores.  64 800 zones of N = 64: 2.6
// ms (5.1 with 28 tiles of 8 x 8 on the wave and the partial sums in LDS, 557
// instructions a step for 344).
//   d, e, reflector i (tau_i in entry i) in row i of qmat; u: see TriArgs.
__global__ __launch_bounds__(64, 3) void k_tridiag64(TriArgs A) {
  __shared__ Tri64 S;
  const int zl = blockIdx.x, lane = threadIdx.x;
  const int64_t z = zone_at(A.zorder, A.z0 + zl);
  if (z < 0) return;
  const int64_t cnt = A.sel_ptr[z + 1] - A.sel_ptr[z];
  if (cnt == 0) return;
  const int n = A.n >= 0 ? A.n : (int)cnt;
  const double* M = A.mat + (size_t)zl * A.zstride;
  double* V = A.qmat + (size_t)zl * A.zstride;
  double* dv = A.dvec + (size_t)zl * A.dz + A.d0;
  double* ev = A.evec + (size_t)zl * A.dz + A.e0;
  double a[64];
#pragma unroll
  for (int c = 0; c < 64; ++c) a[c] = M[(size_t)c * A.ldm + lane];
  double* uz = A.vecs ? A.vecs + (size_t)zl * A.zvec : nullptr;
  const bool has_u = uz != nullptr;
  double u[2] = {0.0, 0.0};
  if (has_u) {
    u[0] = uz[lane];
    u[1] = A.ones >= 0 ? (lane < A.ones ? 1.0 : 0.0) : uz[A.c1 + lane];
  }
  double x = a[0];
#define OAK_TRI(B) tri_steps<B>(S, a, x, u, has_u, n, lane, V, A.ldv, dv, ev, A.dstep);
  OAK_TRI(0) OAK_TRI(1) OAK_TRI(2) OAK_TRI(3) OAK_TRI(4) OAK_TRI(5) OAK_TRI(6) OAK_TRI(7)
#undef OAK_TRI
  if (has_u) {
    uz[lane] = u[0];
    uz[A.c1 + lane] = u[1];
  }
  // rows n - 2 and n - 1 (x: column n - 2; n = 1: column 0), then the identity's
  double dn = a[0];
#pragma unroll
  for (int c = 1; c < 64; ++c) dn = n - 1 == c ? a[c] : dn;
  if (lane == n - 2) dv[lane * A.dstep] = x;
  if (lane == n - 1) {
    if (n >= 2) ev[(n - 2) * A.dstep] = x;
    dv[lane * A.dstep] = dn;
  }
  if (lane >= n) dv[lane * A.dstep] = 1.0;
  if (lane >= n - 1 && lane < 63) ev[lane * A.dstep] = 0.0;
}

void launch_tridiag64(const TriArgs& T, int nzc, hipStream_t st) {
  hipLaunchKernelGGL(k_tridiag64, dim3(nzc), dim3(64), 0, st, T);
}

}  // namespace oakg
