// Launch interfaces of the per-zone analysis kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace oakg {

enum Phase { PH_PREP = 0, PH_SELECT, PH_GRAM, PH_EIG, PH_TMAT, PH_UPDATE, PH_END, PH_COUNT };

// Records an event at each phase boundary; per-phase device time is the sum
// of the intervals that start with a mark of that phase.
struct PhaseTimer {
  hipStream_t st = nullptr;
  std::vector<hipEvent_t> pool;
  std::vector<int> phase;
  size_t used = 0;
  void reset(hipStream_t s) { st = s; used = 0; phase.clear(); }
  void mark(int ph) {
    if (used == pool.size()) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) return;
      pool.push_back(e);
    }
    (void)hipEventRecord(pool[used], st);
    phase.push_back(ph);
    ++used;
  }
  // accumulates milliseconds per phase into ms[PH_COUNT]; call after a sync
  void collect(double* ms) {
    for (int i = 0; i < PH_COUNT; ++i) ms[i] = 0;
    for (size_t i = 0; i + 1 < used; ++i) {
      float t = 0;
      if (hipEventElapsedTime(&t, pool[i], pool[i + 1]) == hipSuccess) ms[phase[i]] += t;
    }
  }
  ~PhaseTimer() {
    for (auto e : pool) (void)hipEventDestroy(e);
  }
};

struct PrepLocArgs {
  int64_t m;
  int N;
  const double* HSf;
  int64_t ldHSf;
  const double *Hxf, *yo, *rmse2;
  const uint8_t* excl;
  double *HS, *innov, *rho;
  unsigned* err;
  double hs_scale;  // HS = hs_scale * HSf (1 for locAnalysis, the inflation for the likelihood)
};

struct PrepEnsArgs {
  int64_t n, m;
  int N;
  const double* E;
  int64_t ldE;
  const int64_t* row_ptr;
  const int32_t* col;
  const double* val;
  const double* Hshift;
  const double *yo, *rmse2;
  const uint8_t* excl;
  double scaling;
  double *HEc, *HS, *innov, *rho;
  unsigned* err;
  // mixed precision (FP32 state): E32, Hshift32 in, HS32 out
  const float* E32;
  const float* Hshift32;
  float* HS32;
};

// The zone at position pos of the zone loop: zones run in the order of
// zorder when the loop has one (zones grouped by observation count), else in
// their own order.
__device__ __forceinline__ int64_t zone_at(const int32_t* __restrict__ zorder, int64_t pos) {
  return zorder ? (int64_t)zorder[pos] : pos;
}

struct ChunkArgs {
  int64_t z0;               // first position of the chunk in the zone loop
  const int32_t* zorder;    // position -> zone, or NULL (position = zone)
  int nzc, N, mode;  // mode 0 = locAnalysis, 1 = ensemble
  int64_t m;
  const int64_t* zone_ptr;
  const int64_t* sel_ptr;
  const int32_t* sel_idx;
  const double* sel_w;
  const double *rho, *innov, *HS;
  double *mat, *ymat, *vec, *ampl;
  double* umat;  // NP = 256: the pole arrays, then T^T (mat: M, then Q F; ymat: the reflectors)
  int32_t* sweeps;
  // 0 = one-sided Jacobi, 1 = Householder tridiagonalisation + functions of T
  int eig_method;
  double *dvec, *evec;      // tridiagonal, NP per zone
  const double* poles;      // the rational approximation's table (poles.hpp)
  unsigned* err;
  double tol;
  int max_sweeps;
  int zone_rows;     // mean rows of a zone
  const double* X0;  // xf (mode 0)
  const double* S;   // Sf (mode 0) or E (mode 1)
  int64_t ldS;
  double* xa;   // mode 0
  double* Out;  // Sa (mode 0) or Ea (mode 1)
  int64_t ldO;
  double scaling, infl, maxcorr;
  const double* maxcorr_v;  // per-element clamp [n] (zone-permuted) or NULL: maxcorr for all
  // mixed precision: 1 = FP32 S (HS32), FP32 members (S32) and FP32 Out32
  int prec;
  const float* HS32;
  const float* S32;
  float* Out32;
  // mode 2 (innovation likelihood and its adjoint): per-zone L, per-zone
  // outputs J_z, dJ/dL_z, dJ/dalpha_z and per-observation dJ/dlog sigma
  const double* corr;
  double *nll_J, *nll_gL, *nll_gA, *nll_gth;
};

// Innovation statistics of report (report.hip): pieces of at most kRepRows
// observations, each inside one observation range.
constexpr int kRepRows = 512;
struct RepPiece {
  int64_t r0, r1;
};
struct ReportArgs {
  int N;
  int layout;  // 0: HS column-major (ldHS); 1: row-major NP-padded in hs_col order
  int64_t npieces;
  int nranges;
  const RepPiece* pieces;
  const int64_t* pbeg;  // [nranges+1] first piece of each range
  const double *d, *rmse2;
  const uint8_t* excl;
  const double* HS;
  const float* HS32;  // layout 1 in FP32 (mixed path)
  int64_t ldHS;
  double* part;   // npieces x (4 + NP)
  double* stats;  // nranges x 5
  unsigned* err;
};

void launch_prep_loc(int NP, const PrepLocArgs& A, hipStream_t st);
void launch_prep_ens(int NP, const PrepEnsArgs& A, hipStream_t st);
void launch_chunk(int NP, const ChunkArgs& A, hipStream_t st, PhaseTimer* tm);
// NP = 128 in two parts (Gram + eigensolve, then transform + update), so
// that the zones solved in observation space can run in between
void launch_solve128(const ChunkArgs& A, hipStream_t st, PhaseTimer* tm);
void launch_apply128(const ChunkArgs& A, hipStream_t st, PhaseTimer* tm);
// zones with 1 <= p < 64 at NP = 128 in observation space (dual.hip): A has
// the dual order and the NP = 64 buffers; ymat128/vec128/ampl receive M^-1/2,
// a, v
void launch_dual128(const ChunkArgs& A, int N, double* ymat128, double* vec128, double* ampl,
                    hipStream_t st, PhaseTimer* tm);
void launch_chunk128(const ChunkArgs& A, hipStream_t st, PhaseTimer* tm);
// NP = 128, 256 (gram_blocks.hip)
void launch_gram_blocks(int NP, const ChunkArgs& A, hipStream_t st);
// NP = 256 (wide256.hip): the whole chunk
void launch_chunk256(const ChunkArgs& A, hipStream_t st, PhaseTimer* tm);
void launch_pole256(const ChunkArgs& A, hipStream_t st);
// A Householder reduction (wide256.hip, tridiag64.hip).  zstride, ldm and ldv: the
// distance between the zones' matrices and the leading dimensions of M and of
// the reflector rows (NP for a zone's own block; a trailing block sits inside
// the zone's reflector block).
// vecs (NULL: none): the zone's vectors (stride zvec) to which the reflectors
// are applied as they are formed, entries 0 .. NP-1 (b, giving Q^T b) and
// c1 .. c1 + NP-1 (1_N for ones >= 0: row r < ones is 1; else as found).
struct TriArgs {
  int64_t z0;
  const int32_t* zorder;
  const int64_t* sel_ptr;
  const double* mat;
  double* qmat;
  int64_t zstride;
  int ldm, ldv;
  // d_i of zone zl at dvec[zl dz + d0 + i dstep], e_i at evec[zl dz + e0 + i dstep]
  double *dvec, *evec;
  int64_t dz, d0, e0, dstep;
  double* vecs;
  int zvec, c1, ones;
  // k_tridiag64: order of the matrix (the rows from it on are the identity's); -1:
  // the zone's observation count
  int n;
};
// up to 64 rows (tridiag64.hip): every step
void launch_tridiag64(const TriArgs& T, int nzc, hipStream_t st);
// Householder reductions on the lower triangle (wide256.hip): d, e, the
// reflectors, and Q^T b and Q^T 1_N (ones = N; -1: the vector in slot 2) in
// place of b and slot 2 of vec
void launch_tridiag_lower128(const ChunkArgs& A, int ones, hipStream_t st);
void launch_tridiag_lower64(const ChunkArgs& A, int ones, hipStream_t st);
// NP = 64, 128 (funcm.hip): the reduction, then M^-1/2 in ymat, a and v;
// dual: the functions of I + G that dual.hip needs
void launch_func(int NP, const ChunkArgs& A, bool dual, hipStream_t st);
// NP = 16, 32: the same, and T = R Omega in place of M (no k_tmat)
void launch_func_small(int NP, const ChunkArgs& A, hipStream_t st);
// the same M^-1/2 from the Jacobi option's eigenvectors
void launch_yyt(int NP, const ChunkArgs& A, hipStream_t st);
// NP = 128: what Omega adds to M^-1/2, for k_update128
void launch_omega_rows128(const ChunkArgs& A, hipStream_t st);
void launch_prep_ens_f32(int NP, const PrepEnsArgs& A, hipStream_t st);
// N <= 128 (update.hip): T from mat (N <= 32) or M^-1/2 from ymat
void launch_update(int NP, const ChunkArgs& A, hipStream_t st);
// N <= 64: Gram, factor and adjoint in one; N > 64: factor and adjoint after the Gram
void launch_nll_chol(int NP, const ChunkArgs& A, hipStream_t st);
void launch_nll128(const ChunkArgs& A, hipStream_t st);
void launch_report(int NP, const ReportArgs& A, hipStream_t st);
void launch_nll_totals(int64_t nz, const double* Jz, const double* gA, double* out,
                       hipStream_t st);

}  // namespace oakg
