// Gram of N > 64 (rrsqrt.F90:135 and the S^T R^-1 d factor of :142): M = I +
// S^T diag(r) S and b = S^T (r o d).
#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"

namespace oakg {

namespace {

// The lower triangle of M in 64 x 64 blocks: NP / 64 (NP / 64 - 1) / 2 off the
// diagonal (16 tiles of 16 x 16) and the diagonal ones in pairs (20 tiles, and b
// for their columns), a workgroup each.  It runs over all the zone's
// observations, four per MFMA step and wave, pipelined as in k_gram.  A block's
// tile J holds its columns 16 J + j for N <= 128 (whose rows of S are stored so
// that a lane's columns are together, hs_col) and 4 j + J above: a lane's four
// columns are one 16-byte load (two in FP64).  MFMA and vector instructions share
// the issue: large blocks keep the latter few (a conversion and half a product
// per MFMA).  grid (zones, parts): neighbouring zones read the same columns of S
// at a time (with a zone's parts one after another N = 256 took a fifth longer).
// One wave per workgroup; four that share the observations (SPLIT, their tiles
// added up through LDS) for zones of kSplitRows or more, so that a few zones with
// many rows fill the device.  The zone's own count decides, not the number of
// zones: its sums keep their order in every schedule.  Each of the two launches
// skips the other's zones, the long ones run first.
// 16 200 zones of 2100 observations, N = 256, FP32: 37.9 ms (blocks of 32 x 32: 49;
// the MFMAs alone 31 at 2.4 GHz).  64 800 zones of N = 128, 14 million rows in
// all: 5.65 ms (a wave per two tile rows, all columns loaded by each: 6.6; with
// kSplitRows 256 and 128: 5.8 and 6.1, 0.01 ms less for 5760 zones of 271 rows).
// What is padding is left out: at N <= 128 the tile rows of the last block beyond
// the members (NL of them hold some), above the
// blocks without members (5760 zones of N = 100, whole analysis 3.57 -> 3.51 ms).
constexpr int kGramSplit = 4, kSplitRows = 512;

template <int NP>
__device__ __forceinline__ int block_col(int X, int J, int j) {
  return 64 * X + (NP == 128 ? 16 * J + j : 4 * j + J);
}

template <int NP, typename TS, bool DIAG, int SPLIT, int NL>
__device__ __forceinline__ void gram_block(int X, int Y, int64_t p0, int pn,
                                             const int32_t* __restrict__ sel_idx,
                                             const double* __restrict__ sel_w, unsigned m,
                                             const double* __restrict__ rho,
                                             const double* __restrict__ innov,
                                             const TS* __restrict__ HS, double* __restrict__ M,
                                             double* __restrict__ bv_out, unsigned* __restrict__ err) {
  constexpr int NT = DIAG ? 10 + NL * (NL + 1) / 2 : 4 * NL;
  typedef TS TS4 __attribute__((ext_vector_type(4)));
  const int part = SPLIT > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int lane = threadIdx.x & 63, kq = lane >> 4, jl = lane & 15;
  d4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = d4{0, 0, 0, 0};
  double bacc[DIAG ? 8 : 1] = {};
  const int nsteps = (pn + 3) >> 2;
  const int32_t* si = sel_idx + p0;
  const double* sw = sel_w + p0;
  struct Stage {
    unsigned l;
    double w, rh, inn;
    TS4 x, y;  // the lane's columns of blocks X and Y
  };
  bool bad = false;  // an index outside 0..m-1 (reported once, after the loop)
  auto fetch_idx = [&](int s, Stage& a) {
    const int q = 4 * s + kq;
    const unsigned qc = q < pn ? q : pn - 1;  // p >= 1 here
    a.l = si[qc];
    a.w = sw[qc];
  };
  const TS* hx = HS + (NP == 128 ? 8 * jl + 4 * X : 64 * X + 4 * jl);
  const TS* hy = HS + (NP == 128 ? 8 * jl + 4 * Y : 64 * Y + 4 * jl);
  auto fetch_row = [&](Stage& a) {
    const bool in = a.l < m;
    bad = bad | !in;
    const unsigned l = in ? a.l : 0;
    a.rh = rho[l];
    if (DIAG) a.inn = innov[l];
    a.x = *reinterpret_cast<const TS4*>(hx + (size_t)l * NP);
    a.y = *reinterpret_cast<const TS4*>(hy + (size_t)l * NP);
  };
  auto step = [&](int s, Stage& c, Stage& n) {
    fetch_row(n);
    const double w = c.w;
    fetch_idx(s + 2 * SPLIT, c);
    asm volatile("" ::: "memory");  // compiler barrier: keeps the loads above here
    const double r = 4 * s + kq < pn ? (w * w) * c.rh : 0.0;
    double x[4], y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      x[k] = (double)c.x[k];
      y[k] = (double)c.y[k];
    }
    int t = 0;
    if constexpr (DIAG) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int I = 0; I < (h ? NL : 4); ++I) {
          const double a = r * (h ? y[I] : x[I]);
#pragma unroll
          for (int J = 0; J <= I; ++J) {
            acc[t] = mfma_f64(a, h ? y[J] : x[J], acc[t]);
            ++t;
          }
        }
      const double rd = r * c.inn;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        bacc[k] = fma(rd, x[k], bacc[k]);
        if (k < NL) bacc[(DIAG ? 4 : 0) + k] = fma(rd, y[k], bacc[(DIAG ? 4 : 0) + k]);
      }
    } else {
#pragma unroll
      for (int I = 0; I < NL; ++I) {
        const double a = r * x[I];
#pragma unroll
        for (int J = 0; J < 4; ++J) {
          acc[t] = mfma_f64(a, y[J], acc[t]);
          ++t;
        }
      }
    }
  };
  Stage A, B;
  fetch_idx(part, A);
  fetch_idx(part + SPLIT, B);
  fetch_row(A);
  int s = part;
  for (; s + SPLIT < nsteps; s += 2 * SPLIT) {
    step(s, A, B);
    step(s + SPLIT, B, A);
  }
  if (s < nsteps) step(s, A, B);
  if (bad) atomicOr(err, OAKG_DERR_IDX);
  if constexpr (SPLIT > 1) {
    __shared__ double red[SPLIT - 1][256];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (part > 0)
#pragma unroll
        for (int q = 0; q < 4; ++q) red[part > 0 ? part - 1 : 0][4 * lane + q] = acc[t][q];
      lds_barrier();
      if (part == 0)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int w = 0; w < SPLIT - 1; ++w) acc[t][q] += red[w][4 * lane + q];
      lds_barrier();
    }
    if constexpr (DIAG) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (part > 0) red[part > 0 ? part - 1 : 0][lane] = bacc[k];
        lds_barrier();
        if (part == 0)
#pragma unroll
          for (int w = 0; w < SPLIT - 1; ++w) bacc[k] += red[w][lane];
        lds_barrier();
      }
    }
    if (part > 0) return;
  }
  // element (i, j) of tile (I, J): i = kq + 4 q in register q, j = jl
  if constexpr (DIAG) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const double b = sum_xor32(sum_xor16(bacc[k]));
      if (lane < 16) bv_out[block_col<NP>(k < 4 ? X : Y, k & 3, lane)] = b;
    }
    // a diagonal block's tile gives both triangles (of a tile (I, I) its own
    // lower half), so that M is exactly symmetric
    int t = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int I = 0; I < 4; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int i = kq + 4 * q, j = jl;
            if (I != J || i >= j) {
              const int gi = block_col<NP>(h ? Y : X, I, i), gj = block_col<NP>(h ? Y : X, J, j);
              const double v = (t < NT ? acc[t < NT ? t : 0][q] : 0.0) + (gi == gj ? 1.0 : 0.0);
              M[(size_t)gi * NP + gj] = v;
              M[(size_t)gj * NP + gi] = v;
            }
          }
          ++t;
        }
  } else if constexpr (NP == 128) {
#pragma unroll
    for (int I = 0; I < 4; ++I)
#pragma unroll
      for (int J = 0; J < 4; ++J)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int gi = block_col<NP>(X, I, kq + 4 * q), gj = block_col<NP>(Y, J, jl);
          const double v = I < NL ? acc[I < NL ? 4 * I + J : 0][q] : 0.0;
          M[(size_t)gi * NP + gj] = v;
          M[(size_t)gj * NP + gi] = v;
        }
  } else {
    // four columns (rows of the mirrored block) of a lane are consecutive
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int gi = 64 * X + 4 * (kq + 4 * q), gj = 64 * Y + 4 * jl;
#pragma unroll
      for (int I = 0; I < 4; ++I) {
        d4 v, u;
#pragma unroll
        for (int J = 0; J < 4; ++J) {
          v[J] = acc[4 * I + J][q];
          u[J] = acc[4 * J + I][q];
        }
        *reinterpret_cast<d4*>(M + (size_t)(gi + I) * NP + gj) = v;
        *reinterpret_cast<d4*>(M + (size_t)(gj + I) * NP + gi) = u;
      }
    }
  }
}

}  // namespace

template <int NP, typename TS, int SPLIT, int NL>
__global__ __launch_bounds__(64 * SPLIT, 2) void k_gram_blocks(int64_t z0, int N,
                                                              const int32_t* __restrict__ zorder,
                                                              const int64_t* __restrict__ sel_ptr,
                                                              const int32_t* __restrict__ sel_idx,
                                                              const double* __restrict__ sel_w, int64_t m,
                                                              const double* __restrict__ rho,
                                                              const double* __restrict__ innov,
                                                              const TS* __restrict__ HS,
                                                              double* __restrict__ mat,
                                                              double* __restrict__ vec,
                                                              unsigned* __restrict__ err) {
  constexpr int NBL = NP / 64, NOFF = NBL * (NBL - 1) / 2, PARTS = NOFF + NBL / 2;
  const int zl = blockIdx.x, y = blockIdx.y;
  const int64_t z = zone_at(zorder, z0 + zl);
  if (z < 0) return;  // the zone is solved by the other pipeline
  const int64_t p0 = sel_ptr[z];
  const int64_t p = sel_ptr[z + 1] - p0;
  if ((p >= kSplitRows) != (SPLIT > 1)) return;  // the other launch's
  double* M = mat + (size_t)zl * NP * NP;
  double* bv_out = vec + (size_t)zl * 4 * NP;
  if (p == 0) {  // M = I, b = 0 (a share of each part)
    constexpr int SH = NP * NP / PARTS;
    for (int e = threadIdx.x; e < SH; e += 64 * SPLIT) {
      const int g = y * SH + e;
      M[g] = (g / NP == g % NP) ? 1.0 : 0.0;
    }
    if (y == 0)
      for (int e = threadIdx.x; e < NP; e += 64 * SPLIT) bv_out[e] = 0.0;
    return;
  }
  if (y < NOFF) {
    const int X = y < 1 ? 1 : (y < 3 ? 2 : 3), Y = y - (y < 1 ? 0 : (y < 3 ? 1 : 3));
    if (64 * X >= N) {  // padding
      for (int e = threadIdx.x; e < 64 * 64; e += 64 * SPLIT) {
        const int i = 64 * X + (e >> 6), j = 64 * Y + (e & 63);
        M[(size_t)i * NP + j] = M[(size_t)j * NP + i] = 0.0;
      }
      return;
    }
    gram_block<NP, TS, false, SPLIT, NL>(X, Y, p0, (int)p, sel_idx, sel_w, (unsigned)m, rho, innov, HS, M,
                                     bv_out, err);
  } else {
    const int X = 2 * (y - NOFF);
    gram_block<NP, TS, true, SPLIT, NL>(X, X + 1, p0, (int)p, sel_idx, sel_w, (unsigned)m, rho, innov, HS, M,
                                    bv_out, err);
  }
}

template <int NP, typename TS, int NL>
static void gram_blocks_t(const ChunkArgs& A, const TS* HS, hipStream_t st) {
  constexpr int NBL = NP / 64, PARTS = NBL * (NBL - 1) / 2 + NBL / 2;
  const dim3 grid(A.nzc, PARTS);
  hipLaunchKernelGGL((k_gram_blocks<NP, TS, kGramSplit, NL>), grid, dim3(64 * kGramSplit), 0, st, A.z0, A.N,
                     A.zorder, A.sel_ptr, A.sel_idx, A.sel_w, A.m, A.rho, A.innov, HS, A.mat, A.vec,
                     A.err);
  hipLaunchKernelGGL((k_gram_blocks<NP, TS, 1, NL>), grid, dim3(64), 0, st, A.z0, A.N, A.zorder, A.sel_ptr,
                     A.sel_idx, A.sel_w, A.m, A.rho, A.innov, HS, A.mat, A.vec, A.err);
}

template <typename TS>
static void gram128_t(const ChunkArgs& A, const TS* HS, hipStream_t st) {
  switch ((A.N - 49) / 16) {  // 65..80, ..96, ..112, ..128 members
    case 1: gram_blocks_t<128, TS, 1>(A, HS, st); break;
    case 2: gram_blocks_t<128, TS, 2>(A, HS, st); break;
    case 3: gram_blocks_t<128, TS, 3>(A, HS, st); break;
    default: gram_blocks_t<128, TS, 4>(A, HS, st); break;
  }
}

void launch_gram_blocks(int NP, const ChunkArgs& A, hipStream_t st) {
  if (NP == 128 && A.prec == 1)
    gram128_t<float>(A, A.HS32, st);
  else if (NP == 128)
    gram128_t<double>(A, A.HS, st);
  else if (A.prec == 1)
    gram_blocks_t<256, float, 4>(A, A.HS32, st);
  else
    gram_blocks_t<256, double, 4>(A, A.HS, st);
}

}  // namespace oakg
