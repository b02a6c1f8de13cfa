// Device helpers shared by the kernels of the zones' matrix functions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"

namespace oakg {

__device__ __forceinline__ double wave_sum_d(double s) { return wave_sum_fast(s); }

// 1/sqrt(h) to full double precision: the hardware estimate y (relative
// error below 2^-22) and one third-order correction, y (1 + e/2 + 3e^2/8)
// with e = 1 - h y^2 (the neglected term 5e^3/16 is below 2^-64)
__device__ __forceinline__ double rsqrt_acc(double h) {
  const double y = __builtin_amdgcn_rsq(h);
  const double e = fma(-h, y * y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}
// 1/x the same way: y (1 + e + e^2) with e = 1 - x y
__device__ __forceinline__ double rcp_acc(double x) {
  const double y = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, y, 1.0);
  return fma(fma(e, e, e), y, y);
}

// Sum over each 16-lane row of a wave, to its lanes.
__device__ __forceinline__ double row_sum16(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x124>(v);
  v += dpp_d<0x128>(v);
  return v;
}

// Sum of a lane's value and that of the lane 16 (32) away, by a row swap in
// registers (a ds_bpermute costs an LDS round trip).
__device__ __forceinline__ double sum_xor16(double v) {
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(v), (unsigned)__double2loint(v), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(v), (unsigned)__double2hiint(v), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}
__device__ __forceinline__ double sum_xor32(double v) {
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(v), (unsigned)__double2loint(v), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(v), (unsigned)__double2hiint(v), false, false);
  return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// Lane c of each 16-lane row, to the row (c constant after unrolling).
__device__ __forceinline__ double row_bcast(double v, int c) {
#define OAK_BC(C) \
  case C: return __builtin_amdgcn_update_dpp(v, v, 0x150 + C, 0xF, 0xF, false);
  switch (c & 15) {
    OAK_BC(0) OAK_BC(1) OAK_BC(2) OAK_BC(3) OAK_BC(4) OAK_BC(5) OAK_BC(6) OAK_BC(7)
    OAK_BC(8) OAK_BC(9) OAK_BC(10) OAK_BC(11) OAK_BC(12) OAK_BC(13) OAK_BC(14)
    default: return __builtin_amdgcn_update_dpp(v, v, 0x15F, 0xF, 0xF, false);
  }
#undef OAK_BC
}

// Orders a wave's own LDS accesses (they complete in order; the compiler must
// not move them across).
__device__ __forceinline__ void lds_fence() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}

// Padded index of row r in the LDS row vectors of the Householder
// reductions: one pad entry per 8 rows (register tiles start every 8 rows).
__host__ __device__ constexpr int tri_rx(int r) { return r + (r >> 3); }

// Entry r of reflector k (zero up to row k, tau_k in entry k) as the N = 256
// reduction leaves them in the zone's block V: rows 0..127 in full, then those
// of the trailing 128 rows in a 128 x 128 block from row 192 (their entries
// below row 128 do not exist: some entry of the block stands in).
__device__ __forceinline__ const double* reflector256(const double* V, int k, int r) {
  return k < 128 ? V + k * 256 + r : V + 192 * 256 + (k - 128) * 128 + (r < 128 ? 0 : r - 128);
}

// What k_pole256 leaves for the products that form F at N > 128, in doubles of a
// zone: the arrays of a block of poles (in a matrix of their own), and, after T_b,
// the weights and G_hh of each block or the 256 weights of the eigenvectors, and
// the number of blocks (0: eigenvectors).
struct PoleSet256 {
  static constexpr int kArrays = 4 * 256 * 32, kWeights = 16 * 136, kCount = kWeights + 256;
};

// T = R Omega (below) with R v = kappa 1, kappa = 1 / |M^1/2 1|, and R 1 known: row c
// of T is T[c][s] = R[c][s] + p_c + q_c v_s for s < N - 1, and T[c][N-1] = p_c + l_c
// (the names as below: p = c1 + c2 wN, q = c3, l = c2).
struct OmegaRow {
  double p, q, l;
};
__device__ __forceinline__ OmegaRow omega_row(int N, double kappa, double r1, double rN, double vN,
                                              double vsum) {
  const double wN = 1.0 / sqrt((double)N);
  const double alv = -1.0 / (fabs(vN) + 1.0), alw = -1.0 / (wN + 1.0);
  const double u2 = wN * (r1 - rN), u3 = vN >= 0 ? kappa + rN : kappa - rN;
  const double c2 = alw * u2 + alv * alw * (wN * vsum) * u3;
  return OmegaRow{fma(c2, wN, kappa * wN), alv * u3, c2};
}

// T = R Omega for the symmetric R = M^-1/2, Omega = RotateVector(w, v) with w =
// 1/sqrt(N) 1 (rrsqrt.F90:185, 737-745; perpSpace matoper.F90:509-535) as the
// identity and rank-one terms, applied to the columns of R that a wave holds in
// MFMA tiles: f[I][r] is R[row(I, r)][c] for the lane's column c and, over the
// four lane groups, all rows.  It becomes X[s][c] = T[c][s]:
//   T[c][s] = R[c][s] (0 at s = N-1) + u1 wN + (alpha_w u2 + alpha_v alpha_w (v.w~)
//             u3) zw_s + alpha_v u3 vt_s,  u1 = (R v)_c, u2 = (R w~)_c, u3 = u1 +
//             sign(v_N) R[c][N-1], zw = w + e_{N-1}, vt = v (0 at N-1), w~ = w (0 at
//             N-1), alpha_v = -1/(|v_N|+1), alpha_w = -1/(wN+1)
template <int NT, typename Row>
__device__ __forceinline__ void omega_columns(d4 (&f)[NT], int N, const double* v, Row row) {
  const double wN = 1.0 / sqrt((double)N), vN = v[N - 1], sgv = vN >= 0 ? 1.0 : -1.0;
  const double alv = -1.0 / (fabs(vN) + 1.0), alw = -1.0 / (wN + 1.0);
  double vw = 0.0, u0 = 0.0, u1 = 0.0, u2 = 0.0;
#pragma unroll
  for (int I = 0; I < NT; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = row(I, r);
      const double vs = s < N ? v[s] : 0.0, x = f[I][r];
      vw += s < N - 1 ? vs : 0.0;
      u1 = fma(x, vs, u1);
      u2 += s < N - 1 ? x : 0.0;
      u0 += s == N - 1 ? x : 0.0;
    }
  vw = wN * sum_xor32(sum_xor16(vw));
  u0 = sum_xor32(sum_xor16(u0));
  u1 = sum_xor32(sum_xor16(u1));
  u2 = wN * sum_xor32(sum_xor16(u2));
  const double u3 = fma(sgv, u0, u1);
  const double c1 = u1 * wN, c2 = alw * u2 + alv * alw * vw * u3, c3 = alv * u3;
#pragma unroll
  for (int I = 0; I < NT; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int s = row(I, r);
      const double zw = s == N - 1 ? wN + 1.0 : wN, vt = s < N - 1 ? v[s] : 0.0;
      const double x = s == N - 1 ? 0.0 : f[I][r];
      f[I][r] = s < N ? x + (c1 + c2 * zw + c3 * vt) : x;
    }
}

}  // namespace oakg
