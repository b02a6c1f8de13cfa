// Innovation negative log-likelihood of the local analysis and its adjoint.
//
// For zone z with local observations q (weights w_q = exp(-(d_q/L_z)^2),
// error variances sigma_q^2, r_q = w_q^2 / sigma_q^2, inflated observation
// anomalies s_q = alpha S_q, innovations d_q) the analysis solves with
// M = I + S'^T diag(r) S', b = S'^T (r o d), a = M^-1 b (rrsqrt.F90:135-142).
// The local innovation covariance D = S' S'^T + diag(1/r) gives, through the
// Woodbury identity and det D = det R det M,
//
//   J_z = 1/2 [ sum_q r_q d_q^2 - b^T a + sum_q log(1/r_q) + log det M ]
//
// (= 1/2 [d^T D^-1 d + log det D]).  Its derivatives, with t_q = s'_q . a and
// u_q = s'_q^T M^-1 s'_q:
//
//   dJ_z/dr_q   = 1/2 [ (d_q - t_q)^2 + u_q - 1/r_q ]
//   dJ_z/dalpha = ( sum_k (1 - 1/mu_k) - a^T a ) / alpha
//
// and r_q = w_q^2 exp(-2 log sigma_q), so dr_q/dlog sigma_q = -2 r_q and
// dr_q/dL_z = r_q (-4 log w_q) / L_z.  u_q is one N x N product
// per observation, the same work as the Gram: |L^-1 s'_q|^2 with M = L L^T.
// The observations with r_q = 0 (excluded) take no part.
//
// A zone with fewer observations than members is solved in observation space: with
// S~ = diag(r)^1/2 S', d~ = diag(r)^1/2 d, D~ = I + S~ S~^T, e~ = D~^-1 d~
//
//   det M = det D~,  sum_q r_q d_q^2 - b^T a = d~^T e~,  a = S~^T e~,
//   sum_k (1 - 1/mu_k) = p - tr D~^-1,  2 r_q dJ_z/dr_q = e~_q^2 - (D~^-1)_qq.
//
// In M's terms the last one is what r (d - t)^2 and r u leave of 1: a precise
// observation's 1 - r u is about 1/mu, and M's own unit eigenvalues are lost in the
// rounding of its large ones.  N = 100, 25 observations with errors of 1e-4 (1e-6) of
// the spread: gradient wrong by 4e-7 (4e-3) of its largest entry with M, by 3e-15
// (4e-15) so.
//
// Rounding moves the eigenvalues of M (D~) by about eps tr M.  Where that is more than 1
// and there are unit eigenvalues (anomalies that sum to zero; two observations of the
// same state), M may be left indefinite, and pivots that are merely raised to 1 let the
// rows of L^-1 grow without bound (infinities, OAKG_ENAN).  A zone with a pivot below
// the noise is factored once more with the noise on its diagonal.
#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"

namespace oakg {

__device__ __forceinline__ double nll_wave_sum(double s) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += shfl_xor_d(s, o);
  return s;
}

constexpr double kNoise = 16 * 0x1p-52;  // of the eigenvalues, in parts of tr M

// A 16 x 16 block by rows, lane i of each 16-lane row holding row i of it in x and of the
// identity in w: eliminated from the top, w becomes L^-1 but for the square roots of
// the pivots.  Exact pivots are at least 1 (M >= I): one that rounding leaves below is
// set to it, as rrsqrt.F90:137 clamps the eigenvalues.  The lane's own pivot: as it was
// found (returned) and as it was used (d).
__device__ __forceinline__ double eliminate16(double (&x)[16], double (&w)[16], int lc, double& d) {
  double own = 1.0;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    double pk = row_bcast(x[k], k);
    own = lc == k ? pk : own;
    pk = pk < 1.0 ? 1.0 : pk;
    const double f = lc > k ? -x[k] * rcp_acc(pk) : 0.0;
#pragma unroll
    for (int c = k + 1; c < 16; ++c) x[c] = fma(f, row_bcast(x[c], k), x[c]);
#pragma unroll
    for (int c = 0; c <= k; ++c) w[c] = fma(f, row_bcast(w[c], k), w[c]);
  }
  d = own < 1.0 ? 1.0 : own;
  return own;
}

// N > 64, zones with N observations or more: one workgroup (4 waves) per zone, after
// k_nll_chol128; wave w takes the observations w, w+4, ... and lane j holds entries j, j+64, ... of the N-vectors.
template <int NP>
__global__ __launch_bounds__(256) void k_nll_adjoint(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                     const int64_t* __restrict__ sel_ptr,
                                                     const int32_t* __restrict__ sel_idx,
                                                     const double* __restrict__ sel_w,
                                                     const double* __restrict__ rho,
                                                     const double* __restrict__ innov,
                                                     const double* __restrict__ HS,
                                                     const double* __restrict__ ymat,
                                                     const double* __restrict__ vec,
                                                     const double* __restrict__ corr, double infl,
                                                     double* __restrict__ Jz,
                                                     double* __restrict__ gL,
                                                     double* __restrict__ gA,
                                                     double* __restrict__ gth) {
  constexpr int KPL = NP / 64;  // vector entries per lane
  __shared__ double sw[4][NP];
  __shared__ double red[4][3];
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  const int64_t p0 = sel_ptr[z];
  const int64_t p = sel_ptr[z + 1] - p0;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (p > 0 && p < N) return;  // in observation space, by k_nll_chol128
  if (p == 0) {
    if (tid == 0) {
      Jz[z] = 0.0;
      gL[z] = 0.0;
      gA[z] = 0.0;
    }
    return;
  }
  const double* V = vec + (size_t)zl * 4 * NP;
  const double* Y = ymat + (size_t)zl * NP * NP;  // W^T: u = |W s|^2
  double ak[KPL];
#pragma unroll
  for (int c = 0; c < KPL; ++c) {
    ak[c] = V[NP + lane + 64 * c];
  }
  const double Lz = corr[z];
  double accL = 0.0, accR = 0.0, accLog = 0.0;
  for (int64_t q = wave; q < p; q += 4) {
    const int64_t l = sel_idx[p0 + q];
    const double w = sel_w[p0 + q];
    const double r = (w * w) * rho[l];
    const double* srow = HS + (size_t)l * NP;
    double t = 0.0;
#pragma unroll
    for (int c = 0; c < KPL; ++c) {
      const int j = lane + 64 * c;
      const double s = srow[hs_col<NP>(j)];
      sw[wave][j] = s;
      t = fma(s, ak[c], t);
    }
    __builtin_amdgcn_wave_barrier();
    t = nll_wave_sum(t);
    double u = 0.0;
#pragma unroll
    for (int c = 0; c < KPL; ++c) {
      const int k = lane + 64 * c;
      double y = 0.0;
      for (int j = 0; j < NP; ++j) y = fma(Y[(size_t)j * NP + k], sw[wave][j], y);
      u = fma(y, y, u);
    }
    u = nll_wave_sum(u);
    __builtin_amdgcn_wave_barrier();
    if (r > 0.0) {
      const double d = innov[l];
      const double e = d - t;
      const double g = 0.5 * (fma(e, e, u) - 1.0 / r);
      if (lane == 0) atomicAdd(gth + l, -2.0 * r * g);
      accL = fma(g * r, -4.0 * log(w) / Lz, accL);
      accR = fma(r * d, d, accR);
      accLog -= log(r);
    }
  }
  if (lane == 0) {
    red[wave][0] = accL;
    red[wave][1] = accR;
    red[wave][2] = accLog;
  }
  __syncthreads();
  if (wave == 0) {
    // log det M, sum_k (1 - 1/mu_k) and b^T a from k_nll_chol128; a^T a
    double aa = 0;
    for (int k = lane; k < NP; k += 64) aa = fma(V[NP + k], V[NP + k], aa);
    aa = nll_wave_sum(aa);
    const double slog = V[3 * NP], sinv = V[3 * NP + 1], ba = V[3 * NP + 2];
    if (lane == 0) {
      const double sL = ((red[0][0] + red[1][0]) + red[2][0]) + red[3][0];
      const double sR = ((red[0][1] + red[1][1]) + red[2][1]) + red[3][1];
      const double sG = ((red[0][2] + red[1][2]) + red[2][2]) + red[3][2];
      Jz[z] = 0.5 * (sR - ba + sG + slog);
      gL[z] = sL;
      gA[z] = (sinv - aa) / infl;
    }
  }
}

// N = 65..128: W = L^-1 of M = L L^T (D~ with p < N, from its Gram tile by tile on)
// by a workgroup per zone, the lower 16 x 16 tiles in LDS (78 KB, two zones a CU).  Block column by block column: the first wave
// eliminates the diagonal tile beside the identity (W_JJ), then MFMA tiles over the
// waves, L_IJ = M_IJ W_JJ^T and M_IK -= L_IJ L_KJ^T; last the columns of W, two a wave,
//   W_IJ = -W_II sum_K L_IK W_KJ.
// W^T to ymat, and for k_nll_adjoint a = W^T W b, log det M, sum (1 - 1/mu) = NP - |W|_F^2
// and b^T a = |W b|^2 to vec; a zone in observation space is finished here.  4096 zones,
// likelihood and gradient with the selection: N = 100, 7 to 53 observations: 0.90 ms (3.9
// with the square root of M from its tridiagonal form), 49 to 280: 8.5 (9.9).
struct Chol128Lds {
  static constexpr int LD = 17;
  double t[36][16 * LD];  // tile (I, J), I >= J, at I (I + 1) / 2 + J: M, then L, W_JJ on the diagonal
  double g[128];          // W b
  double part[4][2];
  double sr[128];         // in observation space: sqrt(r), and the observations
  int l[128];
  double tr, slog;
  int again;
};

__global__ __launch_bounds__(256, 2) void k_nll_chol128(
    int64_t z0, const int32_t* __restrict__ zorder, int N, const int64_t* __restrict__ sel_ptr,
    const int32_t* __restrict__ sel_idx, const double* __restrict__ sel_w, int64_t m,
    const double* __restrict__ rho, const double* __restrict__ innov, const double* __restrict__ HS,
    const double* __restrict__ mat, double* __restrict__ ymat, double* __restrict__ vec,
    const double* __restrict__ corr, double infl, double* __restrict__ Jz, double* __restrict__ gL,
    double* __restrict__ gA, double* __restrict__ gth, unsigned* __restrict__ err) {
  constexpr int NP = 128, NB = 8, LD = Chol128Lds::LD;
  __shared__ Chol128Lds S;
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  const int64_t p0 = sel_ptr[z], p = sel_ptr[z + 1] - p0;
  if (p == 0) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lr = lane >> 4, lc = lane & 15;
  const double* M = mat + (size_t)zl * NP * NP;
  double* Y = ymat + (size_t)zl * NP * NP;
  double* V = vec + (size_t)zl * 4 * NP;
  auto tl = [&](int I, int J) { return S.t[I * (I + 1) / 2 + J]; };
  const bool obs = p < N;
  const int rows = obs ? (int)p : N, nb = obs ? ((int)p + 15) >> 4 : NB;
  double ow = 0.0, orr = 0.0, od = 0.0;  // observation `tid`: weight, r and d
  int ol = 0;
  if (obs && tid < NP) {
    // (beyond the observations: the last one's row, times zero)
    const int64_t q = tid < p ? tid : p - 1;
    ol = sel_idx[p0 + q];
    ow = sel_w[p0 + q];
    const bool bad = ol < 0 || ol >= m;
    if (bad) atomicOr(err, OAKG_DERR_IDX);
    ol = bad ? 0 : ol;
    orr = tid < p && !bad ? (ow * ow) * rho[ol] : 0.0;
    od = tid < p ? innov[ol] : 0.0;
    S.sr[tid] = sqrt(orr);
    S.l[tid] = ol;
  }
  lds_barrier();
  double shift = 0.0;
#pragma unroll 1
  for (int attempt = 0;; ++attempt) {
    if (obs) {
      // D~ = I + S~ S~^T, the tiles over the waves; identity beyond the observations
      int e = 0;
#pragma unroll 1
      for (int I = 0; I < NB; ++I)
#pragma unroll 1
        for (int J = 0; J <= I; ++J, ++e)
          if ((e & 3) == wave) {
            d4 o = {0.0, 0.0, 0.0, 0.0};
            if (I < nb) {
              const double* a = HS + (size_t)S.l[16 * I + lc] * NP + 4 * lr;
              const double* b = HS + (size_t)S.l[16 * J + lc] * NP + 4 * lr;
              const double sa = S.sr[16 * I + lc], sb = S.sr[16 * J + lc];
#pragma unroll 2
              for (int k = 0; k < NP; k += 16) {
                const double2 a0 = *reinterpret_cast<const double2*>(a + k);
                const double2 a1 = *reinterpret_cast<const double2*>(a + k + 2);
                const double2 b0 = *reinterpret_cast<const double2*>(b + k);
                const double2 b1 = *reinterpret_cast<const double2*>(b + k + 2);
                o = mfma_f64(sa * a0.x, sb * b0.x, o);
                o = mfma_f64(sa * a0.y, sb * b0.y, o);
                o = mfma_f64(sa * a1.x, sb * b1.x, o);
                o = mfma_f64(sa * a1.y, sb * b1.y, o);
              }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
              tl(I, J)[(lr + 4 * r) * LD + lc] = o[r] + (I == J && lr + 4 * r == lc ? 1.0 + shift : 0.0);
          }
    } else {
      for (int I = 0; I < NB; ++I)
        for (int J = 0; J <= I; ++J) {
          const int r = tid >> 4, c = tid & 15;
          const double t = M[(size_t)(16 * I + r) * NP + 16 * J + c];
          tl(I, J)[r * LD + c] = t + (I == J && r == c ? shift : 0.0);
        }
    }
    lds_barrier();
    double slog = 0.0, least = HUGE_VAL;
    if (wave == 0 && attempt == 0) {
      double tr = 0.0;
#pragma unroll
      for (int h = 0; h < 2; ++h) tr += tl(4 * h + lr, 4 * h + lr)[lc * LD + lc];
      tr = wave_sum_fast(tr);
      if (lane == 0) S.tr = tr;
    }
#pragma unroll 1
    for (int J = 0; J < nb; ++J) {
      double* D = tl(J, J);
      if (wave == 0) {
        double x[16], w[16], d;
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          x[c] = D[lc * LD + c];
          w[c] = lc == c ? 1.0 : 0.0;
        }
        const double own = eliminate16(x, w, lc, d);
        least = 16 * J + lc < rows ? fmin(least, own) : least;
        const double rs = rsqrt_acc(d);
        slog += log(d);
        if (lr == 0)
#pragma unroll
          for (int c = 0; c < 16; ++c) D[lc * LD + c] = w[c] * rs;
      }
      lds_barrier();
      for (int I = J + 1 + wave; I < nb; I += 4) {
        double* A = tl(I, J);
        d4 o = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q) o = mfma_f64(A[lc * LD + 4 * q + lr], D[lc * LD + 4 * q + lr], o);
        lds_fence();
#pragma unroll
        for (int r = 0; r < 4; ++r) A[(lr + 4 * r) * LD + lc] = o[r];
      }
      lds_barrier();
      int e = 0;
      for (int I = J + 1; I < nb; ++I)
        for (int K = J + 1; K <= I; ++K, ++e)
          if ((e & 3) == wave) {
            const double *A = tl(I, J), *B = tl(K, J);
            double* C = tl(I, K);
            d4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = C[(lr + 4 * r) * LD + lc];
#pragma unroll
            for (int q = 0; q < 4; ++q) o = mfma_f64(-A[lc * LD + 4 * q + lr], B[lc * LD + 4 * q + lr], o);
#pragma unroll
            for (int r = 0; r < 4; ++r) C[(lr + 4 * r) * LD + lc] = o[r];
          }
      lds_barrier();
    }
    if (wave == 0) {
      slog = wave_sum_fast(lr == 0 ? slog : 0.0);
      const double noise = kNoise * S.tr;
      const bool low = __ballot(least < noise) != 0;
      if (lane == 0) {
        S.slog = slog;
        S.again = attempt == 0 && noise > 0x1p-4 && low;
      }
    }
    lds_barrier();
    if (!S.again) break;
    shift = kNoise * S.tr;
    lds_barrier();
  }
  // the columns of W, J and NB - 1 - J for one wave
  double ww = 0.0;
#pragma unroll 1
  for (int h = 0; h < 2; ++h) {
    const int J = h ? NB - 1 - wave : wave;
    d4 w[NB];
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      w[I] = d4{0.0, 0.0, 0.0, 0.0};
      const double* D = tl(I, I);
      if (I == J) {
#pragma unroll
        for (int r = 0; r < 4; ++r) w[I][r] = D[(lr + 4 * r) * LD + lc];
      }
      if (I > J) {
        d4 t = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int K = 0; K < I; ++K)
          if (K >= J) {
            const double* A = tl(I, K);
#pragma unroll
            for (int q = 0; q < 4; ++q) t = mfma_f64(A[lc * LD + 4 * q + lr], w[K][q], t);
          }
#pragma unroll
        for (int q = 0; q < 4; ++q) w[I] = mfma_f64(-D[lc * LD + 4 * q + lr], t[q], w[I]);
      }
    }
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        Y[(size_t)(16 * J + lc) * NP + 16 * I + lr + 4 * r] = w[I][r];
        ww = fma(w[I][r], w[I][r], ww);
      }
  }
  ww = wave_sum_fast(ww);
  __syncthreads();
  double *rhs = S.t[0], *av = S.t[1], *om = S.t[2];  // (the tiles are done)
  if (tid < NP) rhs[tid] = obs ? S.sr[tid] * od : V[tid];
  lds_barrier();
  double ba = 0.0;
  if (tid < NP) {
    double g = 0.0;
    for (int j = 0; j < NP; ++j) g = fma(Y[(size_t)j * NP + tid], rhs[j], g);
    S.g[tid] = g;
    ba = g * g;
  }
  ba = wave_sum_fast(ba);
  if (lane == 0) {
    S.part[wave][0] = ww;
    S.part[wave][1] = ba;
  }
  lds_barrier();
  bool nan = false;
  for (int j = wave; j < NP; j += 4) {
    double a = 0.0, u = 0.0;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const double t = Y[(size_t)j * NP + lane + 64 * c];
      a = fma(t, S.g[lane + 64 * c], a);
      u = fma(t, t, u);
    }
    a = wave_sum_fast(a);
    nan = nan || a != a;
    if (obs) u = wave_sum_fast(u);
    if (lane == 0) {
      av[j] = a;
      om[j] = u;
    }
  }
  if (nan && lane == 0) atomicOr(err, OAKG_DERR_NAN);
  lds_barrier();
  const double sinv = NP - ((S.part[0][0] + S.part[1][0]) + (S.part[2][0] + S.part[3][0]));
  const double sba = (S.part[0][1] + S.part[1][1]) + (S.part[2][1] + S.part[3][1]);
  if (!obs) {
    if (tid < NP) V[NP + tid] = av[tid];
    if (tid == 0) {
      V[3 * NP] = S.slog;
      V[3 * NP + 1] = sinv;
      V[3 * NP + 2] = sba;
    }
    return;
  }
  // observation `tid`, and entry `tid` of a = S~^T e~
  double aa = 0.0, accL = 0.0, accLog = 0.0;
  if (tid < NP) {
    for (int q = 0; q < rows; ++q) aa = fma(S.sr[q] * av[q], HS[(size_t)S.l[q] * NP + tid], aa);
    aa *= aa;
    if (orr > 0.0) {
      const double g2 = om[tid] - av[tid] * av[tid];  // -2 r dJ/dr
      atomicAdd(gth + ol, g2);
      accL = -0.5 * g2 * (-4.0 * log(ow) / corr[z]);
      accLog = -log(orr);
    }
  }
  aa = wave_sum_fast(aa);
  accL = wave_sum_fast(accL);
  accLog = wave_sum_fast(accLog);
  lds_barrier();
  if (lane == 0 && wave < 2) {
    S.g[4 * wave] = aa;
    S.g[4 * wave + 1] = accL;
    S.g[4 * wave + 2] = accLog;
  }
  lds_barrier();
  if (tid == 0) {
    Jz[z] = 0.5 * (sba + (S.g[2] + S.g[6]) + S.slog);
    gL[z] = S.g[1] + S.g[5];
    gA[z] = (sinv - (S.g[0] + S.g[4])) / infl;
  }
}

// After the Gram (gram_blocks.hip): factor and adjoint.
void launch_nll128(const ChunkArgs& A, hipStream_t st) {
  hipLaunchKernelGGL(k_nll_chol128, dim3(A.nzc), dim3(256), 0, st, A.z0, A.zorder, A.N, A.sel_ptr,
                     A.sel_idx, A.sel_w, A.m, A.rho, A.innov, A.HS, A.mat, A.ymat, A.vec, A.corr, A.infl,
                     A.nll_J, A.nll_gL, A.nll_gA, A.nll_gth, A.err);
  hipLaunchKernelGGL(k_nll_adjoint<128>, dim3(A.nzc), dim3(256), 0, st, A.z0, A.zorder, A.N, A.sel_ptr,
                     A.sel_idx, A.sel_w, A.rho, A.innov, A.HS, A.ymat, A.vec, A.corr, A.infl,
                     A.nll_J, A.nll_gL, A.nll_gA, A.nll_gth);
}

// ---------------------------------------------------------------------------
// N <= 64: the zone's Gram, W = L^-1 of M = L L^T (D~ with p < N), and the adjoint in
// one kernel.  J needs log det M and b^T a = |W b|^2, the derivatives M^-1 alone:
// u_q = |W s'_q|^2, a = W^T W b, sum_k (1 - 1/mu_k) = NP - |W|_F^2, so no
// eigenvectors and no square root of M.
//
// M in 16 x 16 tiles (I <= J) in the accumulators; per block J the diagonal
// tile goes to registers by rows (lane i of each 16-lane row of the wave holds
// row i; pivots and pivot rows by DPP broadcast) and is eliminated with the
// identity beside it, which leaves W_JJ, and the rest is MFMA tiles:
//   Z_JK = W_JJ M_JK,  M_IK -= Z_JI^T Z_JK,  W_IJ = -W_II sum_K Z_KI^T W_KJ.
//
// A wave per zone (WPZ = 1), so that all phases of other zones run beside the
// serial elimination of one; four that share the observations (WPZ = 4, the
// elimination by the first) for zones with kShareRows of them or more.  The
// zone's own count decides, so that its sums keep their order in every schedule;
// each of the two launches skips the other's zones.  Bound by
// the MFMAs and the elimination's FP64 issue.  65 536 zones, N = 32, 41
// observations each: 0.69 ms, where the eigensolve by QL, its rotations and the
// adjoint by vector FMAs took 5.9 ms.
// ---------------------------------------------------------------------------
constexpr int kShareRows = 512;

template <int NP, int WPZ>
struct NllLds {
  static constexpr int NB = NP / 16, NT = NB * (NB + 1) / 2, LD = 17;
  double W[NT][16 * LD];  // W_IJ, I >= J, at I (I + 1) / 2 + J
  double tile[16 * LD];
  double bs[NP], gs[NP], as[NP];
  double red[WPZ > 1 ? WPZ - 1 : 1][WPZ > 1 ? 256 : 1];
  double part[WPZ][3], tot[4];
  double noise;  // to be added to the diagonal (0: nothing)
};

// Observation `lane` of a zone solved in observation space: e~ = D~^-1 d~, the diagonal
// of D~^-1, its weight, r and index.
struct ObsSums {
  double e, om, w, r;
  int l;
};

// W, a and the sums of J of a zone, of M + shift I; obs: D~ + shift I and d~ for M and
// b, by the first wave, whose lane q returns observation q's sums.
template <int NP, int WPZ, bool OBS>
__device__ __forceinline__ ObsSums nll_factor(NllLds<NP, WPZ>& S, int N, int64_t p0, int64_t p, double shift,
                                           const int32_t* __restrict__ sel_idx,
                                           const double* __restrict__ sel_w, int64_t m,
                                           const double* __restrict__ rho,
                                           const double* __restrict__ innov,
                                           const double* __restrict__ HS, unsigned* __restrict__ err) {
  using L = NllLds<NP, WPZ>;
  constexpr int NB = L::NB, NT = L::NT, LD = L::LD;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
  auto ut = [](int I, int J) { return J * (J + 1) / 2 + I; };  // I <= J
  auto wt = [](int I, int J) { return I * (I + 1) / 2 + J; };  // I >= J
  const bool obs = OBS && p < N;
  ObsSums o = {0.0, 0.0, 0.0, 0.0, 0};
  bool bad = false;
  d4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
  if (obs) {
    if (wave > 0) return o;
    // ---- D~ = I + S~ S~^T, d~: lane (lr, lc) has columns 16 K + 4 lr .. + 3 of
    // observation 16 I + lc ----
    // (lanes beyond the observations: the last one's row, times zero)
    const int64_t q = lane < p ? lane : p - 1;
    o.l = sel_idx[p0 + q];
    o.w = sel_w[p0 + q];
    bad = o.l < 0 || o.l >= m;
    o.l = bad ? 0 : o.l;
    o.r = lane < p && !bad ? (o.w * o.w) * rho[o.l] : 0.0;
    const double d = lane < p ? innov[o.l] : 0.0;
    const double sr = sqrt(o.r);
    if (lane < NP) S.bs[lane] = sr * d;
    const double* row[NB];
    double sc[NB];
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      row[I] = HS + (size_t)__shfl(o.l, 16 * I + lc) * NP + 4 * lr;
      sc[I] = __shfl(sr, 16 * I + lc);
    }
#pragma unroll 1
    for (int K = 0; K < NB; ++K) {
      double s[NB][4];
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        const double2* r2 = reinterpret_cast<const double2*>(row[I] + 16 * K);
        const double2 t0 = r2[0], t1 = r2[1];
        s[I][0] = sc[I] * t0.x;
        s[I][1] = sc[I] * t0.y;
        s[I][2] = sc[I] * t1.x;
        s[I][3] = sc[I] * t1.y;
      }
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int J = 0; J < NB; ++J)
#pragma unroll
          for (int I = 0; I <= J; ++I) acc[ut(I, J)] = mfma_f64(s[I][c], s[J][c], acc[ut(I, J)]);
    }
    if (__ballot(bad) != 0 && lane == 0) atomicOr(err, OAKG_DERR_IDX);
  } else {
    // ---- M = I + S'^T diag(r) S', b = S'^T (r o d): 16 observations at a time ----
    double bv[NB];
#pragma unroll
    for (int J = 0; J < NB; ++J) bv[J] = 0.0;
    for (int64_t q0 = 16 * wave; q0 < p; q0 += 16 * WPZ) {
      double r[4], rd[4], s[4][NB];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t q = q0 + 4 * i + lr, qc = q < p ? q : p - 1;
        int64_t l = sel_idx[p0 + qc];
        const double w = sel_w[p0 + qc];
        const bool in = l >= 0 && l < m;
        bad = bad || !in;
        l = in ? l : 0;
        const double rr = (w * w) * rho[l], d = innov[l];
        r[i] = q < p && in ? rr : 0.0;
        rd[i] = q < p && in ? rr * d : 0.0;
#pragma unroll
        for (int J = 0; J < NB; ++J) {
          const double t = HS[(size_t)l * NP + 16 * J + lc];
          s[i][J] = q < p && in ? t : 0.0;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int J = 0; J < NB; ++J) {
          bv[J] = fma(rd[i], s[i][J], bv[J]);
#pragma unroll
          for (int I = 0; I <= J; ++I) acc[ut(I, J)] = mfma_f64(r[i] * s[i][I], s[i][J], acc[ut(I, J)]);
        }
    }
    if (__ballot(bad) != 0 && lane == 0) atomicOr(err, OAKG_DERR_IDX);
#pragma unroll
    for (int J = 0; J < NB; ++J) bv[J] = sum_xor32(sum_xor16(bv[J]));
    if (WPZ > 1) {
      // the other waves' parts, tile by tile, to the first
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (wave > 0)
#pragma unroll
          for (int i = 0; i < 4; ++i) S.red[WPZ > 1 ? wave - 1 : 0][4 * lane + i] = acc[t][i];
        lds_barrier();
        if (wave == 0)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int w = 0; w < WPZ - 1; ++w) acc[t][i] += S.red[w][4 * lane + i];
        lds_barrier();
      }
      if (wave > 0 && lr == 0)
#pragma unroll
        for (int J = 0; J < NB; ++J) S.red[WPZ > 1 ? wave - 1 : 0][16 * J + lc] = bv[J];
      lds_barrier();
#pragma unroll
      for (int J = 0; J < NB; ++J)
#pragma unroll
        for (int w = 0; w < WPZ - 1; ++w) bv[J] += S.red[w][16 * J + lc];
    }
    if (wave == 0 && lr == 0)
#pragma unroll
      for (int J = 0; J < NB; ++J) S.bs[16 * J + lc] = bv[J];
  }
  if (wave == 0) {
    // ---- W ----
    double slog = 0.0, least = HUGE_VAL, tr = 0.0;
#pragma unroll
    for (int J = 0; J < NB; ++J)
#pragma unroll
      for (int i = 0; i < 4; ++i) tr += lr + 4 * i == lc ? acc[ut(J, J)][i] : 0.0;
    tr = kNoise * wave_sum_fast(tr);
#pragma unroll
    for (int J = 0; J < NB; ++J) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        S.tile[(lr + 4 * i) * LD + lc] = acc[ut(J, J)][i] + (lr + 4 * i == lc ? 1.0 + shift : 0.0);
      lds_fence();
      double x[16], w[16], d;
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        x[c] = S.tile[lc * LD + c];
        w[c] = lc == c ? 1.0 : 0.0;
      }
      const double own = eliminate16(x, w, lc, d);
      least = 16 * J + lc < (obs ? (int)p : N) ? fmin(least, own) : least;
      const double rs = rsqrt_acc(d);
      slog += log(d);
      if (lr == 0)
#pragma unroll
        for (int c = 0; c < 16; ++c) S.W[wt(J, J)][lc * LD + c] = w[c] * rs;
      lds_fence();
      double wa[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) wa[q] = S.W[wt(J, J)][lc * LD + 4 * q + lr];
#pragma unroll
      for (int K = J + 1; K < NB; ++K) {
        d4 zt = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int q = 0; q < 4; ++q) zt = mfma_f64(wa[q], acc[ut(J, K)][q], zt);
        acc[ut(J, K)] = zt;
      }
#pragma unroll
      for (int K = J + 1; K < NB; ++K)
#pragma unroll
        for (int I = J + 1; I <= K; ++I)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            acc[ut(I, K)] = mfma_f64(-acc[ut(J, I)][q], acc[ut(J, K)][q], acc[ut(I, K)]);
    }
#pragma unroll
    for (int J = 0; J < NB - 1; ++J)
#pragma unroll
      for (int I = J + 1; I < NB; ++I) {
        d4 t = {0.0, 0.0, 0.0, 0.0}, o = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int K = J; K < I; ++K)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            t = mfma_f64(acc[ut(K, I)][q], S.W[wt(K, J)][(4 * q + lr) * LD + lc], t);
#pragma unroll
        for (int q = 0; q < 4; ++q) o = mfma_f64(-S.W[wt(I, I)][lc * LD + 4 * q + lr], t[q], o);
#pragma unroll
        for (int r = 0; r < 4; ++r) S.W[wt(I, J)][(lr + 4 * r) * LD + lc] = o[r];
        lds_fence();
      }
    // ---- W b, a = W^T W b and the sums of J (row or column `lane`) ----
    double g = 0.0, a = 0.0, ww = 0.0;
    const int R = (lane & (NP - 1)) >> 4;
#pragma unroll
    for (int K = 0; K < NB; ++K)
      if (K <= R)
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          const double t = S.W[R * (R + 1) / 2 + K][lc * LD + c];
          g = fma(t, S.bs[16 * K + c], g);
          ww = fma(t, t, ww);
        }
    if (lane < NP) S.gs[lane] = g;
    lds_fence();
#pragma unroll
    for (int I = 0; I < NB; ++I)
      if (I >= R)
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          const double t = S.W[I * (I + 1) / 2 + R][c * LD + lc];
          a = fma(t, S.gs[16 * I + c], a);
          if (OBS) o.om = fma(t, t, o.om);
        }
    o.e = a;
    if (lane < NP) S.as[lane] = a;
    const bool again = shift == 0.0 && tr > 0x1p-4 && __ballot(least < tr) != 0;
    if (a != a && !again) atomicOr(err, OAKG_DERR_NAN);
    slog = lr == 0 ? slog : 0.0;
    slog = wave_sum_fast(slog);
    ww = wave_sum_fast(lane < NP ? 1.0 - ww : 0.0);  // NP - |W|^2 = sum (1 - 1/mu)
    const double aa = wave_sum_fast(lane < NP ? a * a : 0.0);
    const double ba = wave_sum_fast(lane < NP ? g * g : 0.0);
    if (lane == 0) {
      S.tot[0] = slog;
      S.tot[1] = ww;
      S.tot[2] = aa;
      S.tot[3] = ba;
      S.noise = again ? tr : 0.0;
    }
  }
  return o;
}

// One zone, with M + shift I for M.  With shift = 0 and an M that has to be shifted,
// only gL[z] = NaN and gA[z] = the shift are written.
template <int NP, int WPZ, bool OBS>
__device__ __forceinline__ void nll_zone(
    NllLds<NP, WPZ>& S, int N, int64_t z, int64_t p0, int64_t p, double shift,
    const int32_t* __restrict__ sel_idx, const double* __restrict__ sel_w, int64_t m,
    const double* __restrict__ rho, const double* __restrict__ innov, const double* __restrict__ HS,
    const double* __restrict__ corr, double infl, double* __restrict__ Jz, double* __restrict__ gL,
    double* __restrict__ gA, double* __restrict__ gth, unsigned* __restrict__ err) {
  using L = NllLds<NP, WPZ>;
  constexpr int NB = L::NB, NT = L::NT, LD = L::LD;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
  auto wt = [](int I, int J) { return I * (I + 1) / 2 + J; };  // I >= J
  auto sync = [] {
    if (WPZ > 1)
      lds_barrier();
    else
      lds_fence();
  };
  const ObsSums o =
      nll_factor<NP, WPZ, OBS>(S, N, p0, p, shift, sel_idx, sel_w, m, rho, innov, HS, err);
  sync();
  if (S.noise != 0.0) {
    if (threadIdx.x == 0) {
      gL[z] = __builtin_nan("");
      gA[z] = S.noise;
    }
    return;
  }
  const double Lz = corr[z];
  if (OBS && p < N) {
    if (wave > 0) return;
    // ---- observation `lane`, and |a|^2 = |S~^T e~|^2 (entry lane % NP, the
    // observations over the lanes beyond) ----
    const double f = o.r > 0.0 ? sqrt(o.r) * o.e : 0.0;
    double t = 0.0;
    for (int q = 0; q < p; q += 64 / NP) {
      const int k = q + lane / NP;
      const int l = __shfl(o.l, k & 63);
      const double fk = __shfl(f, k & 63);
      t = fma(k < p ? fk : 0.0, HS[(size_t)l * NP + (lane & (NP - 1))], t);
    }
#pragma unroll
    for (int h = NP; h < 64; h *= 2) t += shfl_xor_d(t, h);
    const double aa = wave_sum_fast(lane < NP ? t * t : 0.0);
    const double g2 = o.om - o.e * o.e;  // -2 r dJ/dr
    double accL = 0.0, accLog = 0.0;
    if (o.r > 0.0) {
      atomicAdd(gth + o.l, g2);
      accL = -0.5 * g2 * (-4.0 * log(o.w) / Lz);
      accLog = -log(o.r);
    }
    accL = wave_sum_fast(accL);
    accLog = wave_sum_fast(accLog);
    if (lane == 0) {
      Jz[z] = 0.5 * (S.tot[3] + accLog + S.tot[0]);
      gL[z] = accL;
      gA[z] = (S.tot[1] - aa) / infl;
    }
    return;
  }
  // ---- the observations: lane (lr, lc) has columns 16 K + 4 lr .. + 3 of
  // observation q0 + lc ----
  double ar[NB][4], wo[NT][4];
#pragma unroll
  for (int K = 0; K < NB; ++K)
#pragma unroll
    for (int q = 0; q < 4; ++q) ar[K][q] = S.as[16 * K + 4 * lr + q];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) wo[t][q] = S.W[t][lc * LD + 4 * lr + q];
  double accL = 0.0, accR = 0.0, accLog = 0.0;
  for (int64_t q0 = 16 * wave; q0 < p; q0 += 16 * WPZ) {
    const int64_t q = q0 + lc, qc = q < p ? q : p - 1;
    int64_t l = sel_idx[p0 + qc];
    const double w = sel_w[p0 + qc];
    const bool in = q < p && l >= 0 && l < m;
    l = in ? l : 0;
    const double rr = rho[l], d = innov[l];
    double s[NB][4];
#pragma unroll
    for (int K = 0; K < NB; ++K) {
      const double2* row = reinterpret_cast<const double2*>(HS + (size_t)l * NP + 16 * K + 4 * lr);
      const double2 t0 = row[0], t1 = row[1];
      s[K][0] = t0.x;
      s[K][1] = t0.y;
      s[K][2] = t1.x;
      s[K][3] = t1.y;
    }
    double t = 0.0, u = 0.0;
#pragma unroll
    for (int K = 0; K < NB; ++K)
#pragma unroll
      for (int c = 0; c < 4; ++c) t = fma(s[K][c], ar[K][c], t);
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      d4 y = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int K = 0; K <= I; ++K)
#pragma unroll
        for (int c = 0; c < 4; ++c) y = mfma_f64(wo[wt(I, K)][c], s[K][c], y);
#pragma unroll
      for (int c = 0; c < 4; ++c) u = fma(y[c], y[c], u);
    }
    t = sum_xor32(sum_xor16(t));
    u = sum_xor32(sum_xor16(u));
    const double r = (w * w) * rr;
    if (in && lr == 0 && r > 0.0) {
      const double e = d - t;
      const double g = 0.5 * (fma(e, e, u) - 1.0 / r);
      atomicAdd(gth + l, -2.0 * r * g);
      accL = fma(g * r, -4.0 * log(w) / Lz, accL);
      accR = fma(r * d, d, accR);
      accLog -= log(r);
    }
  }
  accL = wave_sum_fast(accL);
  accR = wave_sum_fast(accR);
  accLog = wave_sum_fast(accLog);
  if (lane == 0) {
    S.part[wave][0] = accL;
    S.part[wave][1] = accR;
    S.part[wave][2] = accLog;
  }
  sync();
  if (threadIdx.x == 0) {
    double s[3] = {S.part[0][0], S.part[0][1], S.part[0][2]};
#pragma unroll
    for (int i = 1; i < WPZ; ++i)
#pragma unroll
      for (int c = 0; c < 3; ++c) s[c] += S.part[i][c];
    Jz[z] = 0.5 * (s[1] - S.tot[3] + s[2] + S.tot[0]);
    gL[z] = s[0];
    gA[z] = (S.tot[1] - S.tot[2]) / infl;
  }
}

#define OAK_NLL_PARAMS                                                                             \
  const int32_t *__restrict__ zorder, const int64_t *__restrict__ sel_ptr,                         \
      const int32_t *__restrict__ sel_idx, const double *__restrict__ sel_w, int64_t m,            \
      const double *__restrict__ rho, const double *__restrict__ innov,                            \
      const double *__restrict__ HS, const double *__restrict__ corr, double infl,                 \
      double *__restrict__ Jz, double *__restrict__ gL, double *__restrict__ gA,                   \
      double *__restrict__ gth, unsigned *__restrict__ err

template <int NP, int WPZ>
__global__ __launch_bounds__(64 * WPZ, 2) void k_nll_chol(int64_t z0, int N, OAK_NLL_PARAMS) {
  __shared__ NllLds<NP, WPZ> S;
  const int64_t z = zone_at(zorder, z0 + blockIdx.x);
  const int64_t p0 = sel_ptr[z], p = sel_ptr[z + 1] - p0;
  if ((p >= kShareRows) != (WPZ > 1)) return;  // the other launch's
  if (p == 0) {
    if (threadIdx.x == 0) Jz[z] = gL[z] = gA[z] = 0.0;
    return;
  }
  nll_zone<NP, WPZ, WPZ == 1>(S, N, z, p0, p, 0.0, sel_idx, sel_w, m, rho, innov, HS, corr, infl, Jz, gL, gA, gth,
                    err);
}

// The zones that have to be shifted, which are rare, found by their marks.  (A second
// factorisation in k_nll_chol, as a loop or as a function, cost it half to all of its
// registers again; N = 16: 75 to 138, N = 64: spills.)
template <int NP>
__global__ __launch_bounds__(256, 2) void k_nll_again(int64_t z0, int nzc, int N, OAK_NLL_PARAMS) {
  __shared__ NllLds<NP, 4> S;
  __shared__ int n, zone[256];
  if (threadIdx.x == 0) n = 0;
  lds_barrier();
  const int k = blockIdx.x * 256 + threadIdx.x;
  if (k < nzc) {
    const int64_t z = zone_at(zorder, z0 + k);
    if (gL[z] != gL[z]) zone[atomicAdd(&n, 1)] = k;
  }
  lds_barrier();
  for (int i = 0; i < n; ++i) {
    const int64_t z = zone_at(zorder, z0 + zone[i]);
    const double shift = gA[z];
    const int64_t p0 = sel_ptr[z], p = sel_ptr[z + 1] - p0;
    lds_barrier();
    nll_zone<NP, 4, true>(S, N, z, p0, p, shift, sel_idx, sel_w, m, rho, innov, HS, corr, infl, Jz, gL, gA, gth,
                    err);
  }
}
#undef OAK_NLL_PARAMS

void launch_nll_chol(int NP, const ChunkArgs& A, hipStream_t st) {
#define OAK_NLL_ARGS                                                                             \
  A.N, A.zorder, A.sel_ptr, A.sel_idx, A.sel_w, A.m, A.rho, A.innov, A.HS, A.corr, A.infl,       \
      A.nll_J, A.nll_gL, A.nll_gA, A.nll_gth, A.err
#define OAK_CHOL_N(P)                                                                            \
  hipLaunchKernelGGL((k_nll_chol<P, 4>), dim3(A.nzc), dim3(256), 0, st, A.z0, OAK_NLL_ARGS);     \
  hipLaunchKernelGGL((k_nll_chol<P, 1>), dim3(A.nzc), dim3(64), 0, st, A.z0, OAK_NLL_ARGS);      \
  hipLaunchKernelGGL(k_nll_again<P>, dim3((A.nzc + 255) / 256), dim3(256), 0, st, A.z0, A.nzc, \
                      OAK_NLL_ARGS)
  switch (NP) {
    case 16: OAK_CHOL_N(16); break;
    case 32: OAK_CHOL_N(32); break;
    case 64: OAK_CHOL_N(64); break;
  }
#undef OAK_CHOL_N
#undef OAK_NLL_ARGS
}

// Sums of the per-zone values (fixed order: one block, strided partial sums
// then a tree) -> out[0] = sum J_z, out[1] = sum dJ/dalpha.
__global__ __launch_bounds__(1024) void k_nll_totals(int64_t nz, const double* __restrict__ Jz,
                                                     const double* __restrict__ gA,
                                                     double* __restrict__ out) {
  __shared__ double sj[1024], sa[1024];
  double a = 0, b = 0;
  for (int64_t z = threadIdx.x; z < nz; z += 1024) {
    a += Jz[z];
    b += gA[z];
  }
  sj[threadIdx.x] = a;
  sa[threadIdx.x] = b;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      sj[threadIdx.x] += sj[threadIdx.x + s];
      sa[threadIdx.x] += sa[threadIdx.x + s];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = sj[0];
    out[1] = sa[0];
  }
}

void launch_nll_totals(int64_t nz, const double* Jz, const double* gA, double* out,
                       hipStream_t st) {
  hipLaunchKernelGGL(k_nll_totals, dim3(1), dim3(1024), 0, st, nz, Jz, gA, out);
}

}  // namespace oakg
