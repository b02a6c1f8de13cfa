// Mixed-precision ensemble analysis (FP32 state): the same steps as the FP64
// path (assimilation.F90:3107-3134, rrsqrt.F90:100-190, assimilation.F90:
// 3299-3320) with FP32 storage of the ensemble, of Ea and of S = H A', and
// the ensemble update A' W on FP32 MFMA.  The N x N eigensolve, the
// eigenvalue functions (1+lambda)^-1 and (1+lambda)^-1/2, the transform T,
// the innovation scaling and the accumulation of S^T R^-1 S stay in FP64.
//
//   k_spmm_obs<float>  HE = H E + Hshift (FP64 accumulation)
//   k_obs_anom_f32     HS = (HE - ybar)/sqrt(N-1) stored FP32, innov/rho FP64
//   k_gram<NP, float>  (analysis.hip; gram_blocks.hip) M = I + S^T diag(r) S
//                      from the FP32 S on FP64 MFMA: products of FP32 values
//                      are exact in FP64, so only the rounding of S to FP32
//                      remains.  An FP32-accumulated Gram has errors of size
//                      eps32 |C| in every direction, including the weakly
//                      observed ones where the analysis keeps the forecast
//                      spread (T ~ I); with |C| up to ~1e5 (precise SSH
//                      observations) that is ~1e-3 of the spread.  Rounding
//                      S itself perturbs those directions only at second order.
//   update             (update.hip for N <= 128)
//                      Ea = xa + sqrt(N-1) infl (Sf T) on v_mfma_f32_16x16x4f32
//                      with T rounded to FP32; xa = xbar + clamp(Sf a) in FP64
//                      (the FP32 sum of N terms Sf_k a_k cancels strongly)
#include "analysis.hpp"
#include "common.hpp"
#include "spmm.hpp"

namespace oakg {

template <int NP, int TR>
__global__ __launch_bounds__(256) void k_obs_anom_f32(int64_t m, int N, const double* __restrict__ HEc,
                                                      const double* __restrict__ yo,
                                                      const double* __restrict__ rmse2,
                                                      const uint8_t* __restrict__ excl,
                                                      double scaling, float* __restrict__ HS,
                                                      double* __restrict__ innov,
                                                      double* __restrict__ rho,
                                                      unsigned* __restrict__ err) {
  __shared__ double tile[TR][NP + 1];
  __shared__ double ybar[TR];
  const int64_t l0 = (int64_t)blockIdx.x * TR;
  for (int e = threadIdx.x; e < TR * NP; e += 256) {
    int k = e / TR, li = e % TR;
    int64_t l = l0 + li;
    tile[li][k] = (l < m && k < N) ? HEc[l + (int64_t)k * m] : 0.0;
  }
  __syncthreads();
  if (threadIdx.x < TR) {
    int li = threadIdx.x;
    int64_t l = l0 + li;
    double s = 0;
    for (int k = 0; k < N; ++k) s += tile[li][k];
    double yb = s / N;
    ybar[li] = yb;
    if (l < m) {
      double r2 = rmse2[l];
      if (!(r2 > 0) || !isfinite(r2)) atomicOr(err, OAKG_DERR_RMSE);
      innov[l] = yo[l] - yb;
      rho[l] = (excl && excl[l]) ? 0.0 : 1.0 / r2;
    }
  }
  __syncthreads();
  const double inv = 1.0 / scaling;
  for (int e = threadIdx.x; e < TR * NP; e += 256) {
    int li = e / NP, k = e % NP;
    int64_t l = l0 + li;
    if (l < m) HS[l * NP + hs_col<NP>(k)] = (k < N) ? (float)((tile[li][k] - ybar[li]) * inv) : 0.0f;
  }
}

static inline unsigned nblk32(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

template <int NP>
static void prep_ens_f32_t(const PrepEnsArgs& A, hipStream_t st) {
  if (A.m == 0) return;
  const SpmmGrid g = spmm_grid(A.m, A.N);
  hipLaunchKernelGGL(k_spmm_obs<float>, dim3(g.x, g.y, g.z), dim3(256), 0, st, A.m, A.n, A.N,
                     A.row_ptr, A.col, A.val, A.E32, A.ldE, A.Hshift32, A.HEc, A.err);
  constexpr int TR = NP > 128 ? 16 : (NP > 64 ? 32 : 64);
  hipLaunchKernelGGL((k_obs_anom_f32<NP, TR>), dim3(nblk32(A.m, TR)), dim3(256), 0, st, A.m, A.N,
                     A.HEc, A.yo, A.rmse2, A.excl, A.scaling, A.HS32, A.innov, A.rho, A.err);
}

void launch_prep_ens_f32(int NP, const PrepEnsArgs& A, hipStream_t st) {
  switch (NP) {
    case 16: prep_ens_f32_t<16>(A, st); break;
    case 32: prep_ens_f32_t<32>(A, st); break;
    case 64: prep_ens_f32_t<64>(A, st); break;
    case 128: prep_ens_f32_t<128>(A, st); break;
    case 256: prep_ens_f32_t<256>(A, st); break;
  }
}

}  // namespace oakg
