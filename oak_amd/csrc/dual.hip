// The analysis of a lightly observed zone (1 <= p < 64 local observations,
// N = 65..128 members) in observation space.  With S~ = diag(sqrt(r)) S the
// p x N weighted anomalies (r = w^2 / sigma^2, rrsqrt.F90:135) and
// d~ = sqrt(r) (yo - Hxf), the ensemble-space matrix is M = I + S~^T S~ and
// b = S~^T d~.  Its N - p eigenvalues beyond the rank of S~ are exactly 1,
// and every output of analysisIncrement is a matrix function of M, so it
// follows from the p x p matrix G = S~ S~^T = U diag(lambda) U^T
// (mu = 1 + lambda):
//
//   a        = M^-1 b        = S~^T (I + G)^-1 d~
//   M^-1/2                   = I - S~^T f(I + G) S~,  f(x) = 1 / (x + sqrt x)
//   M^1/2 1_N                = 1_N + S~^T h(I + G) S~ 1_N,  h(x) = 1 / (1 + sqrt x)
//
// (M^-1/2 - I and M^1/2 - I restricted to the range of S~^T; f and h are
// (1 - x^-1/2) / (x - 1) and (x^1/2 - 1) / (x - 1) written without the
// cancellation at x -> 1).  I + G runs through the NP = 64 reduction and
// k_func with the weights of f and h (funcm.hip), and k_dual_lift writes a,
// the normalised M^1/2 1_N = v, M^-1/2 and its products with 1_N and v into the
// zone's NP = 128 slots, as k_func leaves them for the other zones.  The work per zone drops from that
// of a 128 x 128 reduction to a 64 x 64 one plus two products of 128 x p with
// p x p and p x 128.
//
//   k_dual_gram   M_d = I + G (64 x 64), b_d = d~, S~ 1_N (p rows of HS
//                 gathered and scaled in LDS, 4 x 4 register blocks of G per
//                 thread)
//   k_dual_lift   a, M^1/2 1_N, M^-1/2 from f(I + G) and the two vectors
#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"

namespace oakg {

namespace {

constexpr int PD = 64;        // observation-space size of the dual zones
constexpr int NPP = 128;      // ensemble-space size (NP of the primal slots)
constexpr int LDS_S = NPP + 1;  // padded row of S~ in LDS (rows 2 dwords apart in banks)

// Row q < p of S~ (natural column order) into s[q][*]; rows p..PD-1 zero.
// Returns the scaled innovation d~_q through dq (thread q < PD).
template <typename TS>
__device__ __forceinline__ void load_rows(double (*s)[LDS_S], double* dq, int64_t p0, int64_t p,
                                          const int32_t* __restrict__ sel_idx,
                                          const double* __restrict__ sel_w, int64_t m,
                                          const double* __restrict__ rho,
                                          const double* __restrict__ innov,
                                          const TS* __restrict__ HS, unsigned* __restrict__ err,
                                          double* sr) {
  const int tid = threadIdx.x;
  if (tid < PD) {
    double srq = 0.0, d = 0.0;
    if (tid < p) {
      const int64_t l = sel_idx[p0 + tid];
      if (l < 0 || l >= m) {
        atomicOr(err, OAKG_DERR_IDX);
      } else {
        const double w = sel_w[p0 + tid];
        srq = sqrt((w * w) * rho[l]);
        d = srq * innov[l];
      }
    }
    sr[tid] = srq;
    dq[tid] = d;
  }
  lds_barrier();
  // 128 consecutive stored values per row: position k holds column
  // 16 (k & 7) + (k >> 3) (hs_col<128>)
  for (int e = tid; e < PD * NPP; e += 256) {
    const int q = e >> 7, k = e & 127;
    double v = 0.0;
    if (q < p && sr[q] != 0.0) {
      const int64_t l = sel_idx[p0 + q];
      v = sr[q] * (double)HS[(size_t)l * NPP + k];
    }
    s[q][16 * (k & 7) + (k >> 3)] = v;
  }
  lds_barrier();
}

}  // namespace

template <typename TS>
__global__ __launch_bounds__(256) void k_dual_gram(int64_t z0, const int32_t* __restrict__ zorder,
                                                   const int64_t* __restrict__ sel_ptr,
                                                   const int32_t* __restrict__ sel_idx,
                                                   const double* __restrict__ sel_w, int64_t m,
                                                   const double* __restrict__ rho,
                                                   const double* __restrict__ innov,
                                                   const TS* __restrict__ HS,
                                                   double* __restrict__ mat_d,
                                                   double* __restrict__ vec_d, int N,
                                                   unsigned* __restrict__ err) {
  __shared__ double s[PD][LDS_S];
  __shared__ double dq[PD], sr[PD];
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;  // not a dual zone
  const int64_t p0 = sel_ptr[z];
  const int64_t p = sel_ptr[z + 1] - p0;
  load_rows<TS>(s, dq, p0, p, sel_idx, sel_w, m, rho, innov, HS, err, sr);
  const int tid = threadIdx.x;
  // G[q][k] for q in 4 qb .. 4 qb + 3, k in 4 kb .. 4 kb + 3; the sums run in
  // column order, so G[q][k] and G[k][q] are the same sum (symmetric bits)
  const int qb = tid >> 4, kb = tid & 15;
  double acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0;
  for (int c = 0; c < NPP; ++c) {
    double a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] = s[4 * qb + i][c];
#pragma unroll
    for (int j = 0; j < 4; ++j) b[j] = s[4 * kb + j][c];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = fma(a[i], b[j], acc[i][j]);
  }
  double* Md = mat_d + (size_t)zl * PD * PD;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int q = 4 * qb + i, k = 4 * kb + j;
      Md[q * PD + k] = acc[i][j] + (q == k ? 1.0 : 0.0);
    }
  if (tid < PD) {
    double a = 0.0;
    for (int c = 0; c < N; ++c) a += s[tid][c];
    vec_d[(size_t)zl * 4 * PD + tid] = dq[tid];
    vec_d[(size_t)zl * 4 * PD + 2 * PD + tid] = a;
  }
}

// M^-1/2 = I - S~^T (f S~) on v_mfma_f64_16x16x4f64: wave w forms tile columns
// w and w + 4 of Z = f S~ (its accumulators are the B operands of the second
// product), with the zone's p rows only.  TS is the type of S and of M^-1/2.
template <typename TS>
__global__ __launch_bounds__(256, 2) void k_dual_lift(int64_t z0, const int32_t* __restrict__ zorder,
                                                      int N, const int64_t* __restrict__ sel_ptr,
                                                      const int32_t* __restrict__ sel_idx,
                                                      const double* __restrict__ sel_w, int64_t m,
                                                      const double* __restrict__ rho,
                                                      const double* __restrict__ innov,
                                                      const TS* __restrict__ HS,
                                                      const double* __restrict__ ymat_d,
                                                      const double* __restrict__ vec_d,
                                                      double* __restrict__ ymat,
                                                      double* __restrict__ vec,
                                                      double* __restrict__ ampl,
                                                      unsigned* __restrict__ err) {
  __shared__ double s[PD][LDS_S];
  __shared__ double dq[PD], sr[PD], red[4];
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;
  const int64_t p0 = sel_ptr[z];
  const int64_t p = sel_ptr[z + 1] - p0;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane >> 4, lc = lane & 15;
  const double* F = ymat_d + (size_t)zl * PD * PD;
  const double* Vd = vec_d + (size_t)zl * 4 * PD;  // [PD..2PD) (I+G)^-1 d~, [2PD..3PD) h S~ 1
  load_rows<TS>(s, dq, p0, p, sel_idx, sel_w, m, rho, innov, HS, err, sr);
  const int ni = ((int)p + 15) >> 4, nk = ((int)p + 3) >> 2;  // row tiles, k-steps (p < 64)
  d4 zt[2][4];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj)
#pragma unroll
    for (int I = 0; I < 4; ++I) zt[jj][I] = d4{0.0, 0.0, 0.0, 0.0};
  for (int k = 0; k < nk; ++k) {
    const double b0 = s[4 * k + lr][16 * wave + lc], b1 = s[4 * k + lr][16 * (wave + 4) + lc];
#pragma unroll
    for (int I = 0; I < 4; ++I)
      if (I < ni) {
        const double fv = F[(16 * I + lc) * PD + 4 * k + lr];
        zt[0][I] = mfma_f64(fv, b0, zt[0][I]);
        zt[1][I] = mfma_f64(fv, b1, zt[1][I]);
      }
  }
  TS* R = reinterpret_cast<TS*>(ymat + (size_t)zl * NPP * NPP);
  double s0 = 0.0, s1 = 0.0;  // M^-1/2 1_N of the wave's columns
#pragma unroll 1
  for (int I = 0; I < 8; ++I) {
    d4 x0 = {0.0, 0.0, 0.0, 0.0}, x1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int K = 0; K < 4; ++K)
      if (K < ni) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const double av = s[16 * K + 4 * q + lr][16 * I + lc];
          x0 = mfma_f64(av, zt[0][K][q], x0);
          x1 = mfma_f64(av, zt[1][K][q], x1);
        }
      }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * I + lr + 4 * r, c0 = 16 * wave + lc, c1 = c0 + 64;
      const double y0 = (row == c0 ? 1.0 : 0.0) - x0[r], y1 = (row == c1 ? 1.0 : 0.0) - x1[r];
      R[(size_t)row * NPP + c0] = (TS)y0;
      R[(size_t)row * NPP + c1] = (TS)y1;
      s0 += row < N ? y0 : 0.0;
      s1 += row < N ? y1 : 0.0;
    }
  }
  s0 = sum_xor32(sum_xor16(s0));
  s1 = sum_xor32(sum_xor16(s1));
  double* V = vec + (size_t)zl * 4 * NPP;
  // a, M^1/2 1_N (rows i < 128, threads 0..127; the other waves add zeros)
  const int i = tid;
  double vr = 0.0, ar = 0.0;
  if (tid < NPP) {
    for (int q = 0; q < p; ++q) {
      ar = fma(s[q][i], Vd[PD + q], ar);
      vr = fma(s[q][i], Vd[2 * PD + q], vr);
    }
    vr += i < N ? 1.0 : 0.0;
  }
  const double ss = wave_sum_fast(vr * vr);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  if (lr == 0) {
    V[16 * wave + lc] = s0;
    V[16 * wave + lc + 64] = s1;
  }
  lds_barrier();
  if (tid < NPP) {
    const double nv = (red[0] + red[1]) + (red[2] + red[3]);
    V[3 * NPP + i] = i < N ? 1.0 / sqrt(nv) : 0.0;  // M^-1/2 v
    V[NPP + i] = ar;
    V[2 * NPP + i] = vr / sqrt(nv);
    if (ampl && i < N) ampl[(size_t)z * N + i] = ar;
    if (ar != ar) atomicOr(err, OAKG_DERR_NAN);
  }
}

void launch_dual128(const ChunkArgs& A, int N, double* ymat128, double* vec128, double* ampl,
                    hipStream_t st, PhaseTimer* tm) {
  if (tm) tm->mark(PH_GRAM);
  if (A.prec == 1)
    hipLaunchKernelGGL(k_dual_gram<float>, dim3(A.nzc), dim3(256), 0, st, A.z0, A.zorder, A.sel_ptr,
                       A.sel_idx, A.sel_w, A.m, A.rho, A.innov, A.HS32, A.mat, A.vec, N, A.err);
  else
    hipLaunchKernelGGL(k_dual_gram<double>, dim3(A.nzc), dim3(256), 0, st, A.z0, A.zorder, A.sel_ptr,
                       A.sel_idx, A.sel_w, A.m, A.rho, A.innov, A.HS, A.mat, A.vec, N, A.err);
  if (tm) tm->mark(PH_EIG);
  launch_func(PD, A, true, st);
  if (A.prec == 1)
    hipLaunchKernelGGL(k_dual_lift<float>, dim3(A.nzc), dim3(256), 0, st, A.z0, A.zorder, N,
                       A.sel_ptr, A.sel_idx, A.sel_w, A.m, A.rho, A.innov, A.HS32, A.ymat, A.vec,
                       ymat128, vec128, ampl, A.err);
  else
    hipLaunchKernelGGL(k_dual_lift<double>, dim3(A.nzc), dim3(256), 0, st, A.z0, A.zorder, N,
                       A.sel_ptr, A.sel_idx, A.sel_w, A.m, A.rho, A.innov, A.HS, A.ymat, A.vec,
                       ymat128, vec128, ampl, A.err);
}

}  // namespace oakg
