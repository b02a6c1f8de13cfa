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
// per observation, the same work as the Gram: |L^-1 s'_q|^2 for N <= 64,
// |M^-1/2 s'_q|^2 above.  The observations with r_q = 0 (excluded) take no part.
#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"

namespace oakg {

__device__ __forceinline__ double nll_wave_sum(double s) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) s += shfl_xor_d(s, o);
  return s;
}

// One workgroup (4 waves) per zone; wave w takes the observations w, w+4, ...
// and lane j holds entries j, j+64, ... of the N-vectors.
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
  if (p == 0) {
    if (tid == 0) {
      Jz[z] = 0.0;
      gL[z] = 0.0;
      gA[z] = 0.0;
    }
    return;
  }
  const double* V = vec + (size_t)zl * 4 * NP;
  const double* Y = ymat + (size_t)zl * NP * NP;  // M^-1/2: u = |M^-1/2 s|^2
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
    // sum_k log mu_k, sum_k (1 - 1/mu_k) and b^T a from k_func; a^T a
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

void launch_nll_adjoint128(const ChunkArgs& A, hipStream_t st) {
  hipLaunchKernelGGL(k_nll_adjoint<128>, dim3(A.nzc), dim3(256), 0, st, A.z0, A.zorder, A.N, A.sel_ptr,
                     A.sel_idx, A.sel_w, A.rho, A.innov, A.HS, A.ymat, A.vec, A.corr, A.infl,
                     A.nll_J, A.nll_gL, A.nll_gA, A.nll_gth);
}

// ---------------------------------------------------------------------------
// N <= 64: the zone's Gram, W = L^-1 of M = L L^T, and the adjoint in one
// kernel.  J needs log det M and b^T a = |W b|^2, the derivatives M^-1 alone:
// u_q = |W s'_q|^2, a = W^T W b, sum_k (1 - 1/mu_k) = NP - |W|_F^2, so no
// eigenvectors and no square root of M.
//
// M in 16 x 16 tiles (I <= J) in the accumulators; per block J the diagonal
// tile goes to registers by rows (lane i of each 16-lane row of the wave holds
// row i; pivots and pivot rows by DPP broadcast) and is eliminated with the
// identity beside it, which leaves W_JJ, and the rest is MFMA tiles:
//   Z_JK = W_JJ M_JK,  M_IK -= Z_JI^T Z_JK,  W_IJ = -W_II sum_K Z_KI^T W_KJ.
// Exact pivots are at least 1 (M >= I): one that rounding leaves below is set
// to it, as rrsqrt.F90:137 clamps the eigenvalues.
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
__global__ __launch_bounds__(64 * WPZ, 2) void k_nll_chol(
    int64_t z0, const int32_t* __restrict__ zorder, const int64_t* __restrict__ sel_ptr,
    const int32_t* __restrict__ sel_idx, const double* __restrict__ sel_w, int64_t m,
    const double* __restrict__ rho, const double* __restrict__ innov, const double* __restrict__ HS,
    const double* __restrict__ corr, double infl, double* __restrict__ Jz, double* __restrict__ gL,
    double* __restrict__ gA, double* __restrict__ gth, unsigned* __restrict__ err) {
  constexpr int NB = NP / 16, NT = NB * (NB + 1) / 2, LD = 17;
  __shared__ double W[NT][16 * LD];  // W_IJ, I >= J, at I (I + 1) / 2 + J
  __shared__ double tile[16 * LD];
  __shared__ double bs[NP], gs[NP], as[NP];
  __shared__ double red[WPZ > 1 ? WPZ - 1 : 1][WPZ > 1 ? 256 : 1];
  __shared__ double part[WPZ][3], tot[4];
  const int64_t z = zone_at(zorder, z0 + blockIdx.x);
  const int64_t p0 = sel_ptr[z], p = sel_ptr[z + 1] - p0;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
  if ((p >= kShareRows) != (WPZ > 1)) return;  // the other launch's
  if (p == 0) {
    if (threadIdx.x == 0) Jz[z] = gL[z] = gA[z] = 0.0;
    return;
  }
  auto ut = [](int I, int J) { return J * (J + 1) / 2 + I; };  // I <= J
  auto wt = [](int I, int J) { return I * (I + 1) / 2 + J; };  // I >= J
  bool bad = false;
  // ---- M = I + S'^T diag(r) S', b = S'^T (r o d): 16 observations at a time ----
  d4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = d4{0.0, 0.0, 0.0, 0.0};
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
        for (int i = 0; i < 4; ++i) red[WPZ > 1 ? wave - 1 : 0][4 * lane + i] = acc[t][i];
      lds_barrier();
      if (wave == 0)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int w = 0; w < WPZ - 1; ++w) acc[t][i] += red[w][4 * lane + i];
      lds_barrier();
    }
    if (wave > 0 && lr == 0)
#pragma unroll
      for (int J = 0; J < NB; ++J) red[WPZ > 1 ? wave - 1 : 0][16 * J + lc] = bv[J];
    lds_barrier();
#pragma unroll
    for (int J = 0; J < NB; ++J)
#pragma unroll
      for (int w = 0; w < WPZ - 1; ++w) bv[J] += red[w][16 * J + lc];
  }
  if (wave == 0) {
    if (lr == 0)
#pragma unroll
      for (int J = 0; J < NB; ++J) bs[16 * J + lc] = bv[J];
    // ---- W ----
    double slog = 0.0;
#pragma unroll
    for (int J = 0; J < NB; ++J) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        tile[(lr + 4 * i) * LD + lc] = acc[ut(J, J)][i] + (lr + 4 * i == lc ? 1.0 : 0.0);
      lds_fence();
      double x[16], w[16], d = 1.0;
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        x[c] = tile[lc * LD + c];
        w[c] = lc == c ? 1.0 : 0.0;
      }
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        double pk = row_bcast(x[k], k);
        pk = pk < 1.0 ? 1.0 : pk;
        d = lc == k ? pk : d;
        const double f = lc > k ? -x[k] * rcp_acc(pk) : 0.0;
#pragma unroll
        for (int c = k + 1; c < 16; ++c) x[c] = fma(f, row_bcast(x[c], k), x[c]);
#pragma unroll
        for (int c = 0; c <= k; ++c) w[c] = fma(f, row_bcast(w[c], k), w[c]);
      }
      const double rs = rsqrt_acc(d);
      slog += log(d);
      if (lr == 0)
#pragma unroll
        for (int c = 0; c < 16; ++c) W[wt(J, J)][lc * LD + c] = w[c] * rs;
      lds_fence();
      double wa[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) wa[q] = W[wt(J, J)][lc * LD + 4 * q + lr];
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
            t = mfma_f64(acc[ut(K, I)][q], W[wt(K, J)][(4 * q + lr) * LD + lc], t);
#pragma unroll
        for (int q = 0; q < 4; ++q) o = mfma_f64(-W[wt(I, I)][lc * LD + 4 * q + lr], t[q], o);
#pragma unroll
        for (int r = 0; r < 4; ++r) W[wt(I, J)][(lr + 4 * r) * LD + lc] = o[r];
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
          const double t = W[R * (R + 1) / 2 + K][lc * LD + c];
          g = fma(t, bs[16 * K + c], g);
          ww = fma(t, t, ww);
        }
    if (lane < NP) gs[lane] = g;
    lds_fence();
#pragma unroll
    for (int I = 0; I < NB; ++I)
      if (I >= R)
#pragma unroll
        for (int c = 0; c < 16; ++c) a = fma(W[I * (I + 1) / 2 + R][c * LD + lc], gs[16 * I + c], a);
    if (lane < NP) as[lane] = a;
    if (a != a) atomicOr(err, OAKG_DERR_NAN);
    slog = lr == 0 ? slog : 0.0;
    slog = wave_sum_fast(slog);
    ww = wave_sum_fast(lane < NP ? 1.0 - ww : 0.0);  // NP - |W|^2 = sum (1 - 1/mu)
    const double aa = wave_sum_fast(lane < NP ? a * a : 0.0);
    const double ba = wave_sum_fast(lane < NP ? g * g : 0.0);
    if (lane == 0) {
      tot[0] = slog;
      tot[1] = ww;
      tot[2] = aa;
      tot[3] = ba;
    }
  }
  if (WPZ > 1)
    lds_barrier();
  else
    lds_fence();
  // ---- the observations: lane (lr, lc) has columns 16 K + 4 lr .. + 3 of
  // observation q0 + lc ----
  double ar[NB][4], wo[NT][4];
#pragma unroll
  for (int K = 0; K < NB; ++K)
#pragma unroll
    for (int q = 0; q < 4; ++q) ar[K][q] = as[16 * K + 4 * lr + q];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) wo[t][q] = W[t][lc * LD + 4 * lr + q];
  const double Lz = corr[z];
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
    part[wave][0] = accL;
    part[wave][1] = accR;
    part[wave][2] = accLog;
  }
  if (WPZ > 1)
    lds_barrier();
  else
    lds_fence();
  if (threadIdx.x == 0) {
    double s[3] = {part[0][0], part[0][1], part[0][2]};
#pragma unroll
    for (int i = 1; i < WPZ; ++i)
#pragma unroll
      for (int c = 0; c < 3; ++c) s[c] += part[i][c];
    Jz[z] = 0.5 * (s[1] - tot[3] + s[2] + tot[0]);
    gL[z] = s[0];
    gA[z] = (tot[1] - tot[2]) / infl;
  }
}

void launch_nll_chol(int NP, const ChunkArgs& A, hipStream_t st) {
#define OAK_CHOL(P, WPZ)                                                                           \
  hipLaunchKernelGGL((k_nll_chol<P, WPZ>), dim3(A.nzc), dim3(64 * WPZ), 0, st, A.z0, A.zorder,     \
                     A.sel_ptr, A.sel_idx, A.sel_w, A.m, A.rho, A.innov, A.HS, A.corr, A.infl,     \
                     A.nll_J, A.nll_gL, A.nll_gA, A.nll_gth, A.err)
#define OAK_CHOL_N(P) \
  OAK_CHOL(P, 4);     \
  OAK_CHOL(P, 1)
  switch (NP) {
    case 16: OAK_CHOL_N(16); break;
    case 32: OAK_CHOL_N(32); break;
    case 64: OAK_CHOL_N(64); break;
  }
#undef OAK_CHOL_N
#undef OAK_CHOL
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
