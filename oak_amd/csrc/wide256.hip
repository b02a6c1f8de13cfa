// Analysis kernels for ensembles of 129..256 members (NP = 256).
//
// A zone's 256 x 256 matrix is 512 KB in FP64: it fits neither the
// registers of one workgroup nor its LDS, where the N <= 128 kernels keep
// a zone whole, so each phase splits it its own way:
//   gram_blocks.hip  M = I + S~^T S~ and b = S~^T R^-1 d, eight workgroups.
//   k_tridiag_lower<256>  Householder reduction to tridiagonal form (lower, as
//                  dsytd2), steps 0..127, with the lower triangle in 8 x 8
//                  register tiles over 512 threads, one workgroup per zone:
//                  496 tiles hold columns 8..255, and columns 0..7 sit in
//                  LDS for the seven steps that change them; steps 128..253
//                  by k_tridiag_lower<128> and k_tridiag64.
//   funcm.hip      k_pole256: the rational approximation's solves, a and v.
//   k_qapply256    Q F, then Q (Q F)^T = M^-1/2 and Omega, the reflectors in
//                  compact-WY blocks on MFMA, four workgroups per zone, one
//                  64-column block each.
//   k_update256    out = S [T | a] for the zone's rows, eight workgroups per
//                  zone (one 32-column block of T each) on one XCD.
// The operations are those of the N <= 128 path (rrsqrt.F90:100-190 and the
// post-processing of assimilation.F90:3299-3363); only the split of the work
// and the order of the partial sums differ.  k_tridiag_lower<128> and k_tridiag64
// also serve N = 65..128, k_tridiag64 alone N = 33..64.
#include <algorithm>

#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"

namespace oakg {

namespace {
constexpr int NPW = 256;

// Workgroup g of a launch with `parts` workgroups per zone: zone 8 (g / (8
// parts)) + g % 8 and part (g / 8) % parts, so that the parts of a zone follow
// one another on one XCD (workgroups go to the eight XCDs in turn) and share its
// L2.  A grid with the part in y runs them a whole pass over the zones apart.
__device__ __forceinline__ bool zone_part(int parts, int nzc, int& zl, int& part) {
  const int g = blockIdx.x;
  zl = (g / (8 * parts)) * 8 + (g & 7);
  part = (g >> 3) % parts;
  return zl < nzc;
}
inline dim3 zone_parts(int parts, int nzc) { return dim3((unsigned)((nzc + 7) / 8 * 8 * parts)); }
}  // namespace

// ---------------------------------------------------------------------------
// Householder reduction of M (lower, as dsytd2: H_i x = beta e_1 for the
// column below the diagonal) with the lower triangle in registers.  Thread t
// < 496 holds tile (tr, tc), 1 <= tc <= tr <= 31, of 8 x 8 (rows 8 tr.., columns
// 8 tc..), the tile columns in decreasing order so that the active tiles
// (those meeting the trailing block, 8 tc + 7 > i) are always threads
// 0 .. k - 1 and whole waves fall idle as the block shrinks.  A diagonal tile
// holds the full 8 x 8 block.  Columns 0..7 (every row) are in LDS: only
// steps 0..6 change them, and the row threads treat them.
//
// Step i: every wave forms the reflector from column i, which it carries in
// registers (x[h] = A[lane + 64 h][i]), and keeps its own copy of v in LDS.
// A v is summed per row from 32 partial sums: a row r of tile row R >= 1 gets
// the row sums of tiles (R, 1..R-1) and (R, R), the column sums of tiles
// (R+1..31, R) (the upper triangle's part, by symmetry) and the row sum of
// columns 0..7; each tile writes its sums into the slot of its tile column
// (row sums) or tile row (column sums), so every slot has one writer.  Rows
// 0..7 (steps 0..6) take the column sums of the LDS block instead.  Row
// thread r (waves 4..7) forms p_r = tau (A v)_r and its share of v^T p; the
// tiles then apply A -= v w^T + w v^T with w = p - (tau/2)(v^T p) v.  Column
// i+1 as it stands before the update is published by its tile column (or
// the LDS block), and every wave forms its updated value itself.  Two
// barriers per step.  Steps 0..127 run here; the trailing 128 x 128 block
// then goes to the kernels for 128 and 64 rows (fewer registers, four and twelve
// zones per CU through the late, latency-bound steps).
// Output: reflector i in row i of qmat (tau_i in entry i), d and e.
// ---------------------------------------------------------------------------
template <int NP>
struct TriLowerLds {
  static constexpr int PR = (tri_rx(NP - 1) + 2) & ~1;  // padded length of a row vector
  // distance of the slots of part: a wave writes its column sums into the slots
  // of 8 and more consecutive tile rows at the same place, so an odd distance puts
  // these on different banks (at 144 for NP = 128 and 288 for 256, multiples of 16,
  // conflicts were half of all LDS cycles: 16 200 zones of N = 256, 32.5 ms for
  // 27.1)
  static constexpr int PS = tri_rx(NP - 1) + 3;
  static constexpr int NW = NP == 256 ? 8 : 2;           // waves of the workgroup
  static constexpr int NRW = NP / 64;                  // row waves
  double colw[NW][PR];     // each wave's copy of v
  double pub[2][PR];       // column i+1 before step i's update (double-buffered)
  double pw[2][PR];        // p (double-buffered)
  double part[NP / 8][PS]; // slot s of row r: its partial sum of A v
  double l0[NP][9];        // columns 0..7 of every row (steps 0..6)
  double hp[NRW][8];       // the row waves' shares of (A v)_0..7 (steps 0..6)
  double red[2][NRW];      // the row waves' shares of v^T p (double-buffered)
};

template <int NP>
__global__ __launch_bounds__(NP == 256 ? 512 : 128) void k_tridiag_lower(TriArgs A) {
  const double* __restrict__ mat = A.mat;
  double* __restrict__ qmat = A.qmat;
  const int64_t zstride = A.zstride;
  const int ldm = A.ldm, ldv = A.ldv;
  using L = TriLowerLds<NP>;
  constexpr int NH = NP / 64, H = NP / 2, NB = NP / 8;
  constexpr int NT = (NB - 1) * NB / 2;  // register tiles (tile columns 1..NB-1)
  constexpr int BS = 64 * L::NW;         // threads
  __shared__ L S;
  const int zl = blockIdx.x;
  const int64_t z = zone_at(A.zorder, A.z0 + zl);
  if (z < 0) return;
  if (A.sel_ptr[z + 1] == A.sel_ptr[z]) return;
  double* dv = A.dvec + (size_t)zl * A.dz + A.d0;
  double* ev = A.evec + (size_t)zl * A.dz + A.e0;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const bool own = t < NT;
  int tr = NB - 1, tc = NB - 1;
  if (own) {  // ring s = NB - 1 - tc holds the s + 1 tiles of tile column tc
    int s = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
    while (s * (s + 1) / 2 > t) --s;
    while ((s + 1) * (s + 2) / 2 <= t) ++s;
    tc = NB - 1 - s;
    tr = tc + (t - s * (s + 1) / 2);
  }
  const int r0 = 8 * tr, c0 = 8 * tc;
  const int R0 = tri_rx(r0), C0 = tri_rx(c0);  // tri_rx(r0 + ii) = R0 + ii
  const double* M = mat + (size_t)zl * zstride;
  double* V = qmat + (size_t)zl * zstride;
  double a[8][8];
#pragma unroll
  for (int ii = 0; ii < 8; ++ii)
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) a[ii][jj] = own ? M[(size_t)(r0 + ii) * ldm + c0 + jj] : 0.0;
  const int row = t - (BS - NP);  // the last NP threads: row threads
  if (row >= 0) {
#pragma unroll
    for (int c = 0; c < 8; ++c) S.l0[row][c] = M[(size_t)row * ldm + c];
  }
  for (int e = t; e < NB * L::PS; e += BS) (&S.part[0][0])[e] = 0.0;
  double x[NH];
#pragma unroll
  for (int h = 0; h < NH; ++h) x[h] = M[(size_t)(lane + 64 * h) * ldm];  // column 0 (M symmetric)
  // the vectors: vector q in the registers of wave q
  double u[NH];
  double* uz = A.vecs ? A.vecs + (size_t)zl * A.zvec + (wave ? A.c1 : 0) : nullptr;
  const bool has_u = A.vecs && wave < 2;
  if (has_u) {
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      const int r = lane + 64 * h;
      u[h] = wave && A.ones >= 0 ? (r < A.ones ? 1.0 : 0.0) : uz[r];
    }
  }
  __syncthreads();
  auto pick = [&](int h) {
    double v = x[0];
#pragma unroll
    for (int k = 1; k < NH; ++k) v = h == k ? x[k] : v;
    return v;
  };
  double* col = S.colw[wave];
  for (int i = 0; i < H; ++i) {
    const int b = i & 1;
    double* pw = S.pw[b];
    double* pub = S.pub[b];
    // reflector H = I - tau v v^T with H x = beta e_1, x = A[i+1.., i]
    double tau = 0.0, scal = 0.0, beta;
    double v[NH];
    {
      double s = 0.0;
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const int r = lane + 64 * h;
        if (r >= i + 2) s = fma(x[h], x[h], s);
      }
      const int ia = i + 1;
      // with it x^T u over the same rows (v^T u = scal x^T u + u_{i+1}): the
      // sums' latencies overlap
      double su = 0.0;
      if (has_u) {
#pragma unroll
        for (int h = 0; h < NH; ++h)
          if (lane + 64 * h >= i + 2) su = fma(x[h], u[h], su);
        s = wave_sum_d(s);
        su = wave_sum_d(su);
      } else {
        s = wave_sum_d(s);
      }
      const double alpha = readlane_d(pick(ia >> 6), ia & 63);
      const double di = readlane_d(pick(i >> 6), i & 63);
      beta = alpha;
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
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const int r = lane + 64 * h;
        v[h] = r > i + 1 ? x[h] * scal : (r == i + 1 ? 1.0 : 0.0);
        col[tri_rx(r)] = v[h];
      }
      __builtin_amdgcn_wave_barrier();
      if (wave == L::NW - 1) {
#pragma unroll
        for (int h = 0; h < NH; ++h) {
          const int r = lane + 64 * h;
          V[(size_t)i * ldv + r] = r == i ? tau : v[h];
        }
        if (lane == 0) {
          dv[i * A.dstep] = di;
          ev[i * A.dstep] = beta;
        }
      }
      if (has_u) {
        double ua = u[0];
#pragma unroll
        for (int h = 1; h < NH; ++h) ua = (ia >> 6) == h ? u[h] : ua;
        const double f = -tau * fma(scal, su, readlane_d(ua, ia & 63));
#pragma unroll
        for (int h = 0; h < NH; ++h) u[h] = fma(f, v[h], u[h]);
      }
    }
    // partial sums of the tiles (zeros, once, from a tile that left the trailing
    // block)
    const bool act = own && (c0 + 7 > i);
    double vR[8], vC[8];
#pragma unroll
    for (int jj = 0; jj < 8; ++jj) vC[jj] = col[C0 + jj];
#pragma unroll
    for (int ii = 0; ii < 8; ++ii) vR[ii] = col[R0 + ii];
    // (one branch around all sums: their chains of dependent multiply-adds
    // interleave)
    if (own && c0 + 8 > i) {
      if (act) {
        double ps[8];
#pragma unroll
        for (int ii = 0; ii < 8; ++ii) ps[ii] = a[ii][0] * vC[0];
#pragma unroll
        for (int jj = 1; jj < 8; ++jj)
#pragma unroll
          for (int ii = 0; ii < 8; ++ii) ps[ii] = fma(a[ii][jj], vC[jj], ps[ii]);
#pragma unroll
        for (int ii = 0; ii < 8; ++ii) S.part[tc][R0 + ii] = ps[ii];
        if (tr != tc) {
          double cs[8];
#pragma unroll
          for (int jj = 0; jj < 8; ++jj) cs[jj] = a[0][jj] * vR[0];
#pragma unroll
          for (int ii = 1; ii < 8; ++ii)
#pragma unroll
            for (int jj = 0; jj < 8; ++jj) cs[jj] = fma(a[ii][jj], vR[ii], cs[jj]);
#pragma unroll
          for (int jj = 0; jj < 8; ++jj) S.part[tr][C0 + jj] = cs[jj];
        }
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) S.part[tc][R0 + k] = S.part[tr][C0 + k] = 0.0;
      }
      // column i+1 before this step's update, from its tile column
      if (tc == ((i + 1) >> 3)) {
        const int j0 = (i + 1) & 7;
#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
          if (jj == j0) {
#pragma unroll
            for (int ii = 0; ii < 8; ++ii) pub[R0 + ii] = a[ii][jj];
          }
      }
    }
    // columns 0..7 (steps 0..6): the row sums of the LDS block go to slot 0
    // of rows 8..255; its column sums are (A v)_0..7
    if (row >= 0) {
      if (i < 7) {
        const double vr = col[tri_rx(row)];
        double rs = 0.0, hs[8];
#pragma unroll
        for (int c = 0; c < 8; ++c) {
          const double lv = S.l0[row][c];
          rs = fma(lv, col[c], rs);  // tri_rx(c) = c for c < 8
          hs[c] = lv * vr;
        }
        if (row >= 8) S.part[0][tri_rx(row)] = rs;
        if (i + 1 < 8) pub[tri_rx(row)] = S.l0[row][i + 1];
#pragma unroll
        for (int c = 0; c < 8; ++c) hs[c] = wave_sum_d(hs[c]);
        if (lane == 0) {
#pragma unroll
          for (int c = 0; c < 8; ++c) S.hp[row >> 6][c] = hs[c];
        }
      } else if (i == 7) {
        S.part[0][tri_rx(row)] = 0.0;  // the block has left the trailing matrix
      }
    }
    lds_barrier();
    // p = tau A v and the row waves' shares of v^T p
    if (row >= 0) {
      const int rowx = tri_rx(row);
      double s4[4] = {};
      // the slots of a row of the trailing block below the first live tile
      // column are zeros
#pragma unroll
      for (int q0 = 0; q0 < NB; q0 += 4)
        if (8 * q0 + 32 > i) {
#pragma unroll
          for (int q = 0; q < 4; ++q) s4[q] += S.part[q0 + q][rowx];
        }
      double s = (s4[0] + s4[1]) + (s4[2] + s4[3]);
      if (i < 7 && row < 8) {
        if constexpr (NP == 256)
          s = (S.hp[0][row] + S.hp[1][row]) + (S.hp[2][row] + S.hp[3][row]);
        else
          s = S.hp[0][row] + S.hp[1][row];
      }
      const double pr = row > i ? tau * s : 0.0;
      pw[rowx] = pr;
      double vp = col[rowx] * pr;
      vp = wave_sum_d(vp);
      if (lane == 0) S.red[b][row >> 6] = vp;
    }
    lds_barrier();
    // A -= v w^T + w v^T, w = p + K v, K = -tau/2 v^T p
    double vpt;
    if constexpr (NP == 256)
      vpt = (S.red[b][0] + S.red[b][1]) + (S.red[b][2] + S.red[b][3]);
    else
      vpt = S.red[b][0] + S.red[b][1];
    const double K = -0.5 * tau * vpt;
    if (act) {
      double wC[8];
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) wC[jj] = fma(K, vC[jj], pw[C0 + jj]);
#pragma unroll
      for (int ii = 0; ii < 8; ++ii) {
        const double wR = fma(K, vR[ii], pw[R0 + ii]);
#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
          a[ii][jj] = fma(-vR[ii], wC[jj], fma(-wR, vC[jj], a[ii][jj]));
      }
    }
    if (i < 7 && row >= 0) {
      const int rowx = tri_rx(row);
      const double vr = col[rowx], wr = fma(K, vr, pw[rowx]);
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const double vc = col[c], wc = fma(K, vc, pw[c]);
        S.l0[row][c] = fma(-vr, wc, fma(-wr, vc, S.l0[row][c]));
      }
    }
    // column i+1 after the update (v_{i+1} = 1, w_{i+1} = p_{i+1} + K)
    {
      const double w1 = fma(K, 1.0, pw[tri_rx(i + 1)]);
#pragma unroll
      for (int h = 0; h < NH; ++h) {
        const int r = lane + 64 * h;
        const double w = fma(K, v[h], pw[tri_rx(r)]);
        const double nc = fma(-v[h], w1, fma(-w, 1.0, pub[tri_rx(r)]));
        x[h] = r > i ? nc : 0.0;
      }
    }
  }
  // the trailing block [H, NP)^2 after step H - 1 (the tiles of tile rows and
  // columns >= H / 8; both triangles) to the rows from H of the zone's
  // reflector block: NP = 256, as a dense H x H matrix; NP = 128, as row r,
  // column c - H of rows H..
  if (has_u) {
#pragma unroll
    for (int h = 0; h < NH; ++h) uz[lane + 64 * h] = u[h];
  }
  constexpr int LDO = NP == 256 ? H : NP;
  if (own && tc >= H / 8) {
    double* blk = V + (size_t)H * NP;
#pragma unroll
    for (int ii = 0; ii < 8; ++ii)
#pragma unroll
      for (int jj = 0; jj < 8; ++jj) {
        blk[(size_t)(r0 - H + ii) * LDO + (c0 - H + jj)] = a[ii][jj];
        if (tr != tc) blk[(size_t)(c0 - H + jj) * LDO + (r0 - H + ii)] = a[ii][jj];
      }
  }
}

// NP = 128: steps 0..63 on the lower-triangle tiles (two waves, four zones
// per CU); then the trailing 64 x 64 block (rows 64.., columns 0..63 of the
// zone's reflector block) in full by k_tridiag64 (one wave per zone): its reflectors go to columns 64..127 of the same rows
// (their columns 0..63 keep the block's values, which k_func masks: a
// reflector is zero up to its own index), its d, e and vector entries to
// 64..127.  As one kernel on full 8 x 8 tiles (four waves, two zones per CU)
// the reduction of 64 800 zones took 20.5 ms, like this 14.4 ms.
void launch_tridiag_lower128(const ChunkArgs& A, int ones, hipStream_t st) {
  TriArgs T{A.z0, A.zorder, A.sel_ptr, A.mat, A.ymat, (int64_t)128 * 128, 128, 128,
            A.dvec, A.evec, 128, 0, 0, 1, A.vec, 4 * 128, 2 * 128, ones, 128};
  hipLaunchKernelGGL((k_tridiag_lower<128>), dim3(A.nzc), dim3(128), 0, st, T);
  T.mat = A.ymat + 64 * 128;
  T.qmat = A.ymat + 64 * 128 + 64;
  T.d0 = T.e0 = 64;
  T.vecs = A.vec + 64;
  T.ones = -1;
  T.n = ones - 64;
  launch_tridiag64(T, A.nzc, st);
}

// NP = 64 (33 <= N <= 64, and the observation-space zones of N = 128: ones =
// -1): the whole reduction on one wave per zone, of the steps that the order
// (N, or the zone's observations) has.
void launch_tridiag_lower64(const ChunkArgs& A, int ones, hipStream_t st) {
  const TriArgs T{A.z0, A.zorder, A.sel_ptr, A.mat, A.ymat, (int64_t)64 * 64, 64, 64,
                  A.dvec, A.evec, 64, 0, 0, 1, A.vec, 4 * 64, 2 * 64, ones, ones};
  launch_tridiag64(T, A.nzc, st);
}

// ---------------------------------------------------------------------------
// T = R Omega, R = Q F Q^T, F = T^-1/2, in two passes of the same kernel, each
// with the reflectors applied from the left in blocks of 16 in compact WY form
// (LAPACK dlarft / dlarfb; T_b from k_pole256):
//   STEP 1: F from the pole arrays, Y = Q F to mat
//   STEP 2: Y^T, R = Q Y^T, and Omega applied to its columns: X[s][c] = T[c][s]
// Workgroup y of a zone has columns 64 y .. 64 y + 63 (they depend on no
// other columns): wave w tile column J = 4 y + w, 16 tiles of 16 x 16 in its
// accumulators; tiles and blocks of the padding are left out.  The reflector
// block passes through LDS, double-buffered, the next one loaded while the
// current one is applied; one barrier per block.  Two workgroups a CU.
// Bound by the MFMAs, 2 x 17 400 of 16 x 16 x 4 per zone: 16 200 zones take 15.7
// and 15.6 ms, the MFMAs alone 7.5 each.  With k_pole256 (4.4 ms) they replace Q
// formed explicitly, QL iterations, the rotations on Q, an epilogue and Y Y^T,
// which took 107 ms.
// ---------------------------------------------------------------------------
struct QApplyLds {
  static constexpr int LV = 17;  // padded row of Vb
  double vb[2][NPW * LV];        // Vb[r][j]: row r of reflector 16 b + j
  double tb[2][16 * LV];         // T_b
  double v[NPW];
};

// Tile column J of F = T^-1/2 of a zone (k_pole256's arrays in uz, the weights in tz): what
// one block of poles adds to it.  The lower half's columns see the tile rows
// mirrored (k_func): f[I] is tile row I or 15 - I.
__device__ __forceinline__ void add_block256(int J, int nt, int batch, const double* __restrict__ uz,
                                             const double* __restrict__ tz, d4 (&f)[16]) {
  constexpr int NP = NPW, NB = 16;
  const int lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
  const bool low = J >= NB / 2;
  auto row_of = [&](int I) { return low ? NB - 1 - I : I; };
  const double* P = uz + batch * PoleSet256::kArrays;
  const double* wp = tz + PoleSet256::kWeights + 64 * batch;
  const double* al = P + 2 * NP * 32;
  const double* be = P + 3 * NP * 32;
  const int Js = low ? NB - 1 - J : J;
  auto tile_of = [&](int r) { return r < NB / 2 ? r : NB / 2 + NB - 1 - r; };
  auto load4 = [&](const double* a, int row, int h, double* o) {
    const double2* p = reinterpret_cast<const double2*>(a + (size_t)row * 32 + 8 * lr + 4 * h);
    const double2 x0 = p[0], x1 = p[1];
    o[0] = x0.x;
    o[1] = x0.y;
    o[2] = x1.x;
    o[3] = x1.y;
  };
  const int crow = 16 * tile_of(J) + (low ? 15 - lc : lc);
  double w[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) w[q] = wp[8 * lr + q];
  // the tile on the diagonal: outwards from each column's diagonal entry
  // for the lane's eight poles, then the transpose (as in k_func)
  d4 fd;
  {
    double g[8];
    load4(P + NP * 32, crow, 0, g);
    load4(P + NP * 32, crow, 1, g + 4);
#pragma unroll
    for (int q = 0; q < 8; ++q) g[q] *= w[q];
    const int lcs = low ? 15 - lc : lc, lrs = low ? 3 - lr : lr;
    d4 us = {0.0, 0.0, 0.0, 0.0}, ut;
#pragma unroll
    for (int i = 15; i >= 0; --i) {
      if (i % 4 == 3) asm volatile("" ::: "memory");
      double r[8];
      load4(P, 16 * tile_of(J) + i, 0, r);
      load4(P, 16 * tile_of(J) + i, 1, r + 4);
#pragma unroll
      for (int q = 0; q < 8; ++q) g[q] *= i < lcs ? r[q] : 1.0;
      const double sm = sum_xor32(
          sum_xor16(((g[0] + g[1]) + (g[2] + g[3])) + ((g[4] + g[5]) + (g[6] + g[7]))));
      us[i / 4] = (lrs == (i & 3) && i <= lcs) ? sm : us[i / 4];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      ut[r] = low ? us[3 - r] : us[r];
      fd[r] = 4 * r + lr == lc ? 0.0 : ut[r];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) fd = mfma_f64(ut[r], 4 * r + lr == lc ? 1.0 : 0.0, fd);
  }
  double B[8];
  auto column = [&](const double* a) {
    load4(a, crow, 0, B);
    load4(a, crow, 1, B + 4);
#pragma unroll
    for (int q = 0; q < 8; ++q) B[q] *= w[q];
  };
  auto tile = [&](const double* a, int I, d4 acc) {
    const int rI = row_of(I), t16 = 16 * tile_of(rI);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      double av[4], edge[4];
      load4(a, t16 + (rI < NB / 2 ? lc : 15 - lc), h, av);
      load4(al, t16, h, edge);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        acc = mfma_f64(av[q], B[4 * h + q], acc);
        B[4 * h + q] *= edge[q];
      }
    }
    return acc;
  };
  column(be);
#pragma unroll
  for (int I = NB / 2 - 2; I >= 0; --I)  // outside
    if (I < Js && row_of(I) < nt) f[I] = tile(al, I, f[I]);
  column(al);
#pragma unroll
  for (int I = 1; I < NB; ++I) {  // towards the middle, and beyond it
    if (I == NB / 2) {
#pragma unroll
      for (int q = 0; q < 8; ++q) B[q] *= wp[32 + 8 * lr + q];
    }
    if (I > Js && row_of(I) < nt) f[I] = tile(I < NB / 2 ? be : al, I, f[I]);
  }
#pragma unroll
  for (int I = 0; I < NB / 2; ++I)
    if (I == Js) f[I] += fd;
}

// F of a zone of two blocks of poles, or of the eigenvectors in uz, to Y, tile column J
// by one wave (a function of its own: its loops would make k_qapply256 spill).
__device__ __attribute__((noinline)) void deep_f256(int J, int nt, int count, const double* uz,
                                                    const double* tz, double* Y) {
  constexpr int NP = NPW, NB = 16;
  const int lane = threadIdx.x & 63, lr = lane >> 4, lc = lane & 15;
  auto row_of = [&](int I) { return J >= NB / 2 ? NB - 1 - I : I; };
  d4 f[NB];
#pragma unroll
  for (int I = 0; I < NB; ++I) f[I] = d4{0.0, 0.0, 0.0, 0.0};
  if (count == 0) {
#pragma unroll 1
    for (int k = 0; k < NP; k += 4) {
      const double* zk = uz + (size_t)(k + lr) * NP + lc;
      const double b = tz[PoleSet256::kWeights + k + lr] * zk[16 * J];
#pragma unroll
      for (int I = 0; I < NB; ++I)
        if (row_of(I) < nt) f[I] = mfma_f64(zk[16 * row_of(I)], b, f[I]);
    }
  }
#pragma unroll 1
  for (int batch = 0; batch < count; ++batch) add_block256(J, nt, batch, uz, tz, f);
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) Y[(size_t)(16 * row_of(I) + lr + 4 * r) * NP + 16 * J + lc] = f[I][r];
}

template <int STEP>
__global__ __launch_bounds__(256, 2) void k_qapply256(int nzc, int64_t z0,
                                                      const int32_t* __restrict__ zorder,
                                                      int N, const int64_t* __restrict__ sel_ptr,
                                                      const double* __restrict__ qmat,
                                                      const double* __restrict__ tblk,
                                                      double* __restrict__ mat,
                                                      double* __restrict__ umat,
                                                      const double* __restrict__ vec) {
  constexpr int NP = NPW, NB = 16, LV = QApplyLds::LV;
  __shared__ QApplyLds S;
  int zl, y;
  if (!zone_part(4, nzc, zl, y)) return;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const int lr = lane >> 4, lc = lane & 15;
  const int J = 4 * y + wave;  // the wave's tile column
  double* X = umat + (size_t)zl * NP * NP;
  if (sel_ptr[z + 1] == sel_ptr[z]) {
    if (STEP == 2)
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          X[(size_t)(16 * I + lr + 4 * r) * NP + 16 * J + lc] = I == J && lr + 4 * r == lc ? 1.0 : 0.0;
    return;
  }
  const double* V = qmat + (size_t)zl * NP * NP;
  double* Y = mat + (size_t)zl * NP * NP;
  const int nt = (N + 15) >> 4, nblk = N > 2 ? (N + 13) >> 4 : 0;
  // the lower half's columns see the tile rows mirrored (k_func): f[I] is
  // tile row I or NB - 1 - I
  const bool low = STEP == 1 && J >= NB / 2;
  auto row_of = [&](int I) { return low ? NB - 1 - I : I; };
  d4 f[NB];
#pragma unroll
  for (int I = 0; I < NB; ++I) f[I] = d4{0.0, 0.0, 0.0, 0.0};
  if (J < nt) {
    if constexpr (STEP == 1) {
      const double* tz = tblk + (size_t)zl * NP * NP;
      const double* uz = umat + (size_t)zl * NP * NP;
      const int count = __builtin_amdgcn_readfirstlane((int)tz[PoleSet256::kCount]);
      if (count == 1) {
        add_block256(J, nt, 0, uz, tz, f);
      } else {
        deep_f256(J, nt, count, uz, tz, Y);
#pragma unroll
        for (int I = 0; I < NB; ++I)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            f[I][r] = Y[(size_t)(16 * row_of(I) + lr + 4 * r) * NP + 16 * J + lc];
      }
    } else {
      // Y^T: tile (J, I) of Y, transposed by a product with the identity (exact)
#pragma unroll
      for (int I = 0; I < NB; ++I)
        if (I < nt) {
          d4 y;
#pragma unroll
          for (int r = 0; r < 4; ++r) y[r] = Y[(size_t)(16 * J + lr + 4 * r) * NP + 16 * I + lc];
#pragma unroll
          for (int r = 0; r < 4; ++r) f[I] = mfma_f64(y[r], 4 * r + lr == lc ? 1.0 : 0.0, f[I]);
        }
    }
  }
  if (STEP == 2) S.v[t] = t < N ? vec[(size_t)zl * 4 * NP + 2 * NP + t] : 0.0;
  // thread t moves reflector pj of a block, rows pr + 16 e, and entry t of T_b
  const int pj = t >> 4, pr = t & 15;
  double pf[16], pt = 0.0;
  auto load_block = [&](int b) {
#pragma unroll
    for (int e = 0; e < 16; ++e) pf[e] = *reflector256(V, 16 * b + pj, pr + 16 * e);
    pt = tblk[(size_t)zl * NP * NP + b * 136 + (pj <= pr ? pr * (pr + 1) / 2 + pj : 0)];
  };
  if (nblk > 0) load_block(nblk - 1);
#pragma unroll 1
  for (int b = nblk - 1; b >= 0; --b) {
    double* vb = S.vb[b & 1];
    double* tb = S.tb[b & 1];
    const int k = 16 * b + pj;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int r = pr + 16 * e;
      vb[r * LV + pj] = (k < N - 2 && r > k) ? pf[e] : 0.0;
    }
    tb[pj * LV + pr] = pj <= pr ? -pt : 0.0;
    if (b > 0) load_block(b - 1);
    lds_barrier();
    if (J >= nt) continue;
    d4 w = {0.0, 0.0, 0.0, 0.0}, wp = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      const int rI = row_of(I);
      if (rI >= b && rI < nt)
#pragma unroll
        for (int q = 0; q < 4; ++q) w = mfma_f64(vb[(16 * rI + 4 * q + lr) * LV + lc], f[I][q], w);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) wp = mfma_f64(tb[lc * LV + 4 * q + lr], w[q], wp);
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      const int rI = row_of(I);
      if (rI >= b && rI < nt)
#pragma unroll
        for (int q = 0; q < 4; ++q) f[I] = mfma_f64(vb[(16 * rI + lc) * LV + 4 * q + lr], wp[q], f[I]);
    }
  }
  if (STEP == 1) {
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        Y[(size_t)(16 * row_of(I) + lr + 4 * r) * NP + 16 * J + lc] = f[I][r];
    return;
  }
  lds_barrier();
  omega_columns(f, N, S.v, [&](int I, int r) { return 16 * I + lr + 4 * r; });
#pragma unroll
  for (int I = 0; I < NB; ++I)
#pragma unroll
    for (int r = 0; r < 4; ++r) X[(size_t)(16 * I + lr + 4 * r) * NP + 16 * J + lc] = f[I][r];
}

// ---------------------------------------------------------------------------
// Update (update.hip's MODEs) for the zone's rows, transposed on the MFMA.
// Workgroup cb of a zone's eight has columns 32 cb .. 32 cb + 31 of T; they share
// an L2 for the zone's rows of S; 68 KB of LDS each, two per CU.  A strip's members are
// all in registers before the product, which gives the mean of the state
// without a pass of its own; the factors sqrt(N-1) cancel (update.hip).  Each
// workgroup forms S a itself (bit-identical in all eight), for the mean and the
// clamp.  The k index is permuted within pairs of MFMA steps as in k_update64.
// 16 200 zones of 161 rows, FP32 members: 9.6 ms (18 with a mean from a pass of
// its own, a division per element and a third of the MFMAs on the increment).
// TE is the type of S and out (double, or float on the mixed path); the
// products are in FP64.
// ---------------------------------------------------------------------------
template <int MODE, typename TE>
__global__ __launch_bounds__(256, 2) void k_update256(int nzc, int64_t z0,
                                                   const int32_t* __restrict__ zorder, int N,
                                                   const int64_t* __restrict__ zone_ptr,
                                                   const double* __restrict__ umat,
                                                   const double* __restrict__ vec,
                                                   const double* __restrict__ X0,
                                                   const TE* __restrict__ S, int64_t ldS,
                                                   double* __restrict__ xa, TE* __restrict__ Out,
                                                   int64_t ldO, double scaling, double infl,
                                                   double maxcorr,
                                                   const double* __restrict__ maxcorr_v) {
#pragma clang fp contract(off)
  constexpr int NP = NPW, CB = 32, NCB = NP / CB, NBc = CB / 16, LW = NP + 2, Q = NP / 4;
  __shared__ __attribute__((aligned(16))) double Ws[CB * LW];
  __shared__ __attribute__((aligned(16))) double as[NP];
  int zl, cb;
  if (!zone_part(NCB, nzc, zl, cb) || CB * cb >= N) return;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;
  const int64_t i0 = zone_ptr[z];
  const int64_t sz = zone_ptr[z + 1] - i0;
  if (sz <= 0) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int li = lane & 15, kk = lane >> 4;
  const double* X = umat + (size_t)zl * NP * NP + (size_t)CB * cb * NP;  // X[s][k] = T[k][s]
  const double* a = vec + (size_t)zl * 4 * NP + NP;
  copy_batched<16>(threadIdx.x, NP * CB, 256, [&](int e) { return X[e]; },
                   [&](int e, double t) { Ws[(e / NP) * LW + e % NP] = t; });
  as[threadIdx.x] = MODE == 1 ? a[threadIdx.x] / scaling : a[threadIdx.x];
  auto k_of = [&](int q) { return 8 * (q >> 1) + 2 * kk + (q & 1); };
  lds_barrier();
  const double* lw = Ws + li * LW + 2 * kk;
  for (int64_t rb = 16 * wave; rb < sz; rb += 64) {
    const bool rok = rb + li < sz;
    const int64_t row = i0 + (rok ? rb + li : 0);
    TE b[Q];
    {
      // pairs of members on, the last ones clamped to a member that exists
      const TE* p = S + row + (int64_t)(2 * kk) * ldS;
#pragma unroll
      for (int q = 0; q < Q; q += 2) {
        b[q] = p[k_of(q) < N ? 0 : -(int64_t)k_of(q) * ldS];
        b[q + 1] = p[k_of(q + 1) < N ? ldS : -(int64_t)k_of(q) * ldS];
        p += 8 * ldS;
        __builtin_amdgcn_sched_barrier(0);  // addresses as they are needed
      }
    }
    double x0 = 0.0, dx = 0.0;
    if (MODE == 1) {
#pragma unroll
      for (int q = 0; q < Q; ++q) x0 += k_of(q) < N ? (double)b[q] : 0.0;
      x0 = sum_xor32(sum_xor16(x0)) / N;
    } else {
      x0 = X0[row];
    }
    // opaque here: the conversions above would else be kept for below, and spill
#pragma unroll
    for (int q = 0; q < Q; ++q) asm volatile("" : "+v"(b[q]));
    d4 acc[NBc];
#pragma unroll
    for (int J = 0; J < NBc; ++J) acc[J] = d4{0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < Q / 2; ++p) {
      asm volatile("" ::: "memory");  // the reads of later pairs stay below
      double d[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const double s = (double)b[2 * p + h];
        d[h] = rok && k_of(2 * p + h) < N ? (MODE == 1 ? s - x0 : s) : 0.0;
      }
      const double2 ak = *reinterpret_cast<const double2*>(as + 8 * p + 2 * kk);
      dx = fma(d[0], ak.x, dx);
      dx = fma(d[1], ak.y, dx);
      double2 A[NBc];
#pragma unroll
      for (int J = 0; J < NBc; ++J) A[J] = *reinterpret_cast<const double2*>(lw + 16 * J * LW + 8 * p);
#pragma unroll
      for (int J = 0; J < NBc; ++J) acc[J] = mfma_f64(A[J].x, d[0], acc[J]);
#pragma unroll
      for (int J = 0; J < NBc; ++J) acc[J] = mfma_f64(A[J].y, d[1], acc[J]);
    }
    double xar = x0 + sum_xor32(sum_xor16(dx));
    if (MODE == 1) {
      const double mc = maxcorr_v ? maxcorr_v[row] : maxcorr;
      if (xar - mc > x0) xar = x0 + mc;
      if (xar < x0 - mc) xar = x0 - mc;
    }
    if (MODE == 0 && rok && cb == 0 && kk == 0) xa[row] = xar;
#pragma unroll
    for (int J = 0; J < NBc; ++J)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int c = CB * cb + 16 * J + kk + 4 * r;
        if (rok && c < N) {
          const double o = acc[J][r], d = infl != 1.0 ? infl * o : o;
          Out[row + (int64_t)c * ldO] = (TE)(MODE == 1 ? xar + d : o);
        }
      }
  }
}

// ---------------------------------------------------------------------------
void launch_chunk256(const ChunkArgs& A, hipStream_t st, PhaseTimer* tm) {
  if (tm) tm->mark(PH_GRAM);
  launch_gram_blocks(256, A, st);
  if (tm) tm->mark(PH_EIG);
  // the reduction: steps 0..127, then the trailing block (rows 128..191 of
  // the reflectors' matrix, dense) as launch_tridiag_lower128 does, its
  // reflectors to rows 192..255
  constexpr int64_t ZS = (int64_t)256 * 256;
  TriArgs T{A.z0, A.zorder, A.sel_ptr, A.mat, A.ymat, ZS, 256, 256, A.dvec, A.evec, 256, 0, 0, 1,
            A.vec, 4 * 256, 2 * 256, A.N, 256};
  hipLaunchKernelGGL((k_tridiag_lower<256>), dim3(A.nzc), dim3(512), 0, st, T);
  T.mat = A.ymat + 128 * 256;
  T.qmat = A.ymat + 192 * 256;
  T.ldm = T.ldv = 128;
  T.d0 = T.e0 = 128;
  T.vecs = A.vec + 128;
  T.ones = -1;
  hipLaunchKernelGGL((k_tridiag_lower<128>), dim3(A.nzc), dim3(128), 0, st, T);
  T.mat = T.qmat + 64 * 128;
  T.qmat = T.qmat + 64 * 128 + 64;
  T.d0 = T.e0 = 192;
  T.vecs = A.vec + 192;
  T.n = std::max(A.N - 192, 0);
  launch_tridiag64(T, A.nzc, st);
  launch_pole256(A, st);
  const double* tb = A.ymat + 128 * 256;
  hipLaunchKernelGGL(k_qapply256<1>, zone_parts(4, A.nzc), dim3(256), 0, st, A.nzc, A.z0, A.zorder, A.N,
                     A.sel_ptr, A.ymat, tb, A.mat, A.umat, A.vec);
  if (tm) tm->mark(PH_TMAT);
  hipLaunchKernelGGL(k_qapply256<2>, zone_parts(4, A.nzc), dim3(256), 0, st, A.nzc, A.z0, A.zorder, A.N,
                     A.sel_ptr, A.ymat, tb, A.mat, A.umat, A.vec);
  if (tm) tm->mark(PH_UPDATE);
  const dim3 nb = zone_parts(8, A.nzc);
  if (A.prec == 1)
    hipLaunchKernelGGL((k_update256<1, float>), nb, dim3(256), 0, st, A.nzc, A.z0, A.zorder,
                       A.N, A.zone_ptr, A.umat, A.vec, A.X0, A.S32, A.ldS, A.xa, A.Out32, A.ldO,
                       A.scaling, A.infl, A.maxcorr, A.maxcorr_v);
  else if (A.mode == 0)
    hipLaunchKernelGGL((k_update256<0, double>), nb, dim3(256), 0, st, A.nzc, A.z0,
                       A.zorder, A.N, A.zone_ptr, A.umat, A.vec, A.X0, A.S, A.ldS, A.xa, A.Out,
                       A.ldO, A.scaling, A.infl, A.maxcorr, A.maxcorr_v);
  else
    hipLaunchKernelGGL((k_update256<1, double>), nb, dim3(256), 0, st, A.nzc, A.z0,
                       A.zorder, A.N, A.zone_ptr, A.umat, A.vec, A.X0, A.S, A.ldS, A.xa, A.Out,
                       A.ldO, A.scaling, A.infl, A.maxcorr, A.maxcorr_v);
  if (tm) tm->mark(PH_END);
}

}  // namespace oakg
