// The update of a zone's rows for N <= 128:
//   MODE 0 (locAnalysis): xa = xf + Sf a, Sa = Sf T   (rrsqrt.F90:151,185,463)
//   MODE 1 (ensemble): Sf = (E - xbar)/sqrt(N-1) with xbar the members' mean;
//     xa = xbar + clamp(Sf a); Ea = xa + sqrt(N-1) (inflation Sf T)
//     (assimilation.F90:3301-3320).  The factors sqrt(N-1) cancel in Sf T and
//     go to a in Sf a, so that E - xbar is used as it is.
// Computed transposed on the MFMA (A = T^T, B = Sf^T) so that the loads and
// stores of each 16-row strip are 16 consecutive rows of four members.  A
// strip's members are all in registers before the product: the mean of the
// state needs no pass of its own over the ensemble.  FP32 members: E - xbar
// and T rounded to FP32 for v_mfma_f32_16x16x4f32, Sf a in FP64 (the sum of N
// terms Sf_k a_k cancels strongly).
#include <type_traits>

#include "analysis.hpp"
#include "common.hpp"
#include "eigen_common.hpp"

namespace oakg {

namespace {

template <typename T>
using vec4 = typename std::conditional<sizeof(T) == 4, f4, d4>::type;
// D row of register r in lane group kk (the two instructions differ)
template <typename T>
__device__ __forceinline__ constexpr int drow(int kk, int r) {
  return sizeof(T) == 4 ? 4 * kk + r : kk + 4 * r;
}
__device__ __forceinline__ d4 mfma(double a, double b, d4 c) { return mfma_f64(a, b, c); }
__device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The lane's members k(q) = 8 (q / 2) + 2 kk + q % 2 of a row, those past N
// replaced by the first; the addresses are formed as they are needed (all at
// once they spill), and the values made opaque, so that their conversions for
// the mean are not kept for the product.
template <int Q, typename TE>
__device__ __forceinline__ void load_members(TE (&b)[Q], const TE* S, int64_t row, int64_t ldS, int kk,
                                             int N) {
  const TE* p = S + row + (int64_t)(2 * kk) * ldS;
  const TE* first = S + row;
#pragma unroll
  for (int q = 0; q < Q; q += 2) {
    const int k = 4 * q + 2 * kk;
    b[q] = *(k < N ? p : first);
    b[q + 1] = *(k + 1 < N ? p + ldS : first);
    p += 8 * ldS;
    __builtin_amdgcn_sched_barrier(0);
  }
}
template <int Q, typename TE>
__device__ __forceinline__ void opaque(TE (&b)[Q]) {
#pragma unroll
  for (int q = 0; q < Q; ++q) asm volatile("" : "+v"(b[q]));
}

// What the rows of a strip share: the row's mean (or xf), the clamp and the
// column of the increment.  b: the lane's members k(q) of row `row`, replaced
// by the anomalies; as: a (MODE 0) or a / sqrt(N-1).  Returns xa.
template <int Q, int MODE, typename TE, typename K, typename As>
__device__ __forceinline__ double strip_head(TE (&b)[Q], int N, K k, As as, bool rok, int64_t row,
                                             const double* __restrict__ X0, double maxcorr,
                                             const double* __restrict__ maxcorr_v) {
#pragma clang fp contract(off)
  double x0 = 0.0, dx = 0.0;
  if (MODE == 1) {
#pragma unroll
    for (int q = 0; q < Q; ++q) x0 += k(q) < N ? (double)b[q] : 0.0;
    x0 = sum_xor32(sum_xor16(x0)) / N;
    opaque(b);
  } else {
    x0 = X0[row];
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (q % 4 == 0) asm volatile("" ::: "memory");  // a piece by piece
    double d = MODE == 1 ? (double)b[q] - x0 : (double)b[q];
    d = rok && k(q) < N ? d : 0.0;
    dx = fma(d, as(q), dx);
    b[q] = (TE)d;
  }
  double xar = x0 + sum_xor32(sum_xor16(dx));
  if (MODE == 1) {
    const double mc = maxcorr_v ? maxcorr_v[row] : maxcorr;
    if (xar - mc > x0) xar = x0 + mc;
    if (xar < x0 - mc) xar = x0 - mc;
  }
  return xar;
}

template <int MODE, typename TE>
__device__ __forceinline__ TE out_value(double o, double xar, double infl) {
#pragma clang fp contract(off)
  if (MODE == 0) return (TE)o;
  const double d = infl != 1.0 ? infl * o : o;
  return (TE)(xar + d);
}

}  // namespace

// N <= 32: T (left in mat by the eigensolve) in registers, no LDS, no
// barrier; `wpz` waves share a zone's strips, the next strip's members are
// loaded before the current one's product.
template <int NP, int MODE, typename TE>
__global__ __launch_bounds__(256, NP == 32 ? 3 : 4) void k_update_small(int64_t z0, const int32_t* __restrict__ zorder,
                                                         int nzc, int wpz, int N,
                                                         const int64_t* __restrict__ zone_ptr,
                                                         const double* __restrict__ mat,
                                                         const double* __restrict__ vec,
                                                         const double* __restrict__ X0,
                                                         const TE* __restrict__ S, int64_t ldS,
                                                         double* __restrict__ xa,
                                                         TE* __restrict__ Out, int64_t ldO,
                                                         double scaling, double infl, double maxcorr,
                                                         const double* __restrict__ maxcorr_v) {
  constexpr int NB = NP / 16, Q = NP / 4;
  const int wave = blockIdx.x * 4 + (threadIdx.x >> 6), zl = wave / wpz, sub = wave % wpz;
  if (zl >= nzc) return;
  const int64_t z = zone_at(zorder, z0 + zl);
  const int64_t i0 = zone_ptr[z], sz = zone_ptr[z + 1] - i0;
  if (16 * (int64_t)sub >= sz) return;
  const int lane = threadIdx.x & 63, li = lane & 15, kk = lane >> 4;
  TE b[Q], nb[Q];
  auto load = [&](int64_t rb, TE (&v)[Q]) {
    const int64_t row = i0 + (rb + li < sz ? rb + li : 0);
#pragma unroll
    for (int q = 0; q < Q; ++q) v[q] = S[row + (int64_t)(4 * q + kk < N ? 4 * q + kk : 0) * ldS];
  };
  load(16 * sub, b);
  const double* T = mat + (size_t)zl * NP * NP;
  const double* a = vec + (size_t)zl * 4 * NP + NP;
  TE t[NB][Q];
  double as[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    as[q] = MODE == 1 ? a[4 * q + kk] / scaling : a[4 * q + kk];
#pragma unroll
    for (int J = 0; J < NB; ++J) t[J][q] = (TE)T[(4 * q + kk) * NP + 16 * J + li];
  }
  for (int64_t rb = 16 * sub; rb < sz; rb += 16 * wpz) {
    const bool more = rb + 16 * wpz < sz;
    if (more) load(rb + 16 * wpz, nb);
    const bool rok = rb + li < sz;
    const int64_t row = i0 + (rok ? rb + li : 0);
    const double xar = strip_head<Q, MODE>(b, N, [&](int q) { return 4 * q + kk; },
                                           [&](int q) { return as[q]; }, rok, row, X0, maxcorr, maxcorr_v);
    if (MODE == 0 && rok && kk == 0) xa[row] = xar;
    vec4<TE> acc[NB];
#pragma unroll
    for (int J = 0; J < NB; ++J) acc[J] = vec4<TE>{0, 0, 0, 0};
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int J = 0; J < NB; ++J) acc[J] = mfma(t[J][q], b[q], acc[J]);
#pragma unroll
    for (int J = 0; J < NB; ++J)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = 16 * J + drow<TE>(kk, r);
        if (rok && col < N) Out[row + (int64_t)col * ldO] = out_value<MODE, TE>(acc[J][r], xar, infl);
      }
#pragma unroll
    for (int q = 0; q < Q; ++q) b[q] = nb[q];
  }
}

// 33 <= N <= 64: a workgroup per zone forms T = R Omega from M^-1/2 (in ymat)
// in LDS - R is symmetric, so that Omega is applied to its columns and row s
// holds column s of T - and its four waves take the strips in turn.  The k
// index of the MFMA steps is permuted within pairs (lane group kk covers k =
// 8 p + 2 kk and the next), so that one LDS read of two entries serves two
// steps.  Bound by the reads and writes of the ensemble: 64 800 zones of 121 rows,
// N = 64, 8.0 GB and 2.1 GB of M^-1/2, 2.67 ms.  With T from a kernel of its own,
// a spilling product that waited for each load and the mean in a pass before,
// these took 1.6, 10.5 and 0.7 ms.  NB tile rows and columns hold members.
template <int MODE, typename TE, int NB>
__global__ __launch_bounds__(256, 3) void k_update64(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                     const int64_t* __restrict__ sel_ptr,
                                                     const int64_t* __restrict__ zone_ptr,
                                                     const double* __restrict__ ymat,
                                                     const double* __restrict__ vec,
                                                     const double* __restrict__ X0,
                                                     const TE* __restrict__ S, int64_t ldS,
                                                     double* __restrict__ xa, TE* __restrict__ Out,
                                                     int64_t ldO, double scaling, double infl,
                                                     double maxcorr,
                                                     const double* __restrict__ maxcorr_v) {
  constexpr int NP = 64, Q = 4 * NB;
  constexpr int LD = sizeof(TE) == 4 ? NP + 4 : NP + 2;  // reads of 16 rows on distinct banks
  typedef TE TE2 __attribute__((ext_vector_type(2)));
  __shared__ __attribute__((aligned(16))) TE L[NP * LD];
  __shared__ double u[4][NP], w[4][NP], v[NP], as[NP], vws;
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  const int64_t i0 = zone_ptr[z], sz = zone_ptr[z + 1] - i0;
  if (sz <= 0) return;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, li = lane & 15, kk = lane >> 4;
  const double* Vz = vec + (size_t)zl * 4 * NP;
  auto k_of = [&](int q) { return 8 * (q >> 1) + 2 * kk + (q & 1); };
  TE b[Q];
  auto load = [&](int64_t rb) {
    const int64_t row = i0 + (rb + li < sz ? rb + li : 0);
#pragma unroll
    for (int q = 0; q < Q; ++q) b[q] = S[row + (int64_t)(k_of(q) < N ? k_of(q) : 0) * ldS];
  };
  if (sel_ptr[z + 1] == sel_ptr[z]) {  // no observations: T = I, a = 0
    load(16 * wave);
    for (int e = tid; e < NP * NP; e += 256) L[(e / NP) * LD + e % NP] = e / NP == e % NP ? 1 : 0;
    if (tid < NP) as[tid] = 0.0;
    lds_barrier();
  } else {
    // thread (h, r): rows s = 4 i + h of column r (M^-1/2 is symmetric)
    const int r = tid & 63, h = tid >> 6;
    const double* R = ymat + (size_t)zl * NP * NP;
    double x[NP / 4];
#pragma unroll
    for (int i = 0; i < NP / 4; ++i) x[i] = R[(4 * i + h) * NP + r];
    if (tid < NP) {
      as[tid] = MODE == 1 ? Vz[NP + tid] / scaling : Vz[NP + tid];
      v[tid] = tid < N ? Vz[2 * NP + tid] : 0.0;
    }
    lds_barrier();
    // (k_tmat): with zw = w + e_{N-1}, vt = v but 0 at N - 1,
    // T[r][s] = R[r][s] (0 at s = N-1) + u1 w + (alpha_w u2 + alpha_v alpha_w
    // (v.w~) u3) zw_s + alpha_v u3 vt_s, u1 = (R v)_r, u2 = (R w~)_r, u3 = u1 +
    // sign(v_N) R[r][N-1]
    double su = 0.0, sw = 0.0;
#pragma unroll
    for (int i = 0; i < NP / 4; ++i) {
      const int s = 4 * i + h;
      su = fma(x[i], v[s], su);
      sw += s < N - 1 ? x[i] : 0.0;
    }
    u[h][r] = su;
    w[h][r] = sw;
    const double wN = 1.0 / sqrt((double)N), vN = v[N - 1], sgv = vN >= 0 ? 1.0 : -1.0;
    const double alv = -1.0 / (fabs(vN) + 1.0), alw = -1.0 / (wN + 1.0);
    if (wave == 0) {
      const double s = wave_sum_fast(lane < N - 1 ? v[lane] * wN : 0.0);
      if (lane == 0) vws = s;
    }
    load(16 * wave);  // in flight while T is finished (LDS barriers only)
    lds_barrier();
    const double u0 = R[(size_t)(N - 1) * NP + r];
    const double u1 = (u[0][r] + u[1][r]) + (u[2][r] + u[3][r]);
    const double u2 = wN * ((w[0][r] + w[1][r]) + (w[2][r] + w[3][r]));
    const double u3 = fma(sgv, u0, u1);
    const double c1 = u1 * wN, c2 = alw * u2 + alv * alw * vws * u3, c3 = alv * u3;
#pragma unroll
    for (int i = 0; i < NP / 4; ++i) {
      const int s = 4 * i + h;
      const double zw = s == N - 1 ? wN + 1.0 : wN, vt = s < N - 1 ? v[s] : 0.0;
      const double t = s == N - 1 ? 0.0 : x[i];
      L[s * LD + r] = (TE)(s < N ? t + (c1 + c2 * zw + c3 * vt) : x[i]);
    }
    lds_barrier();
  }
  const TE* lt = L + li * LD + 2 * kk;
  for (int64_t rb = 16 * wave; rb < sz; rb += 64) {
    if (rb != 16 * wave) load(rb);
    const bool rok = rb + li < sz;
    const int64_t row = i0 + (rok ? rb + li : 0);
    const double xar = strip_head<Q, MODE>(b, N, k_of, [&](int q) { return as[k_of(q)]; }, rok, row, X0,
                                           maxcorr, maxcorr_v);
    if (MODE == 0 && rok && kk == 0) xa[row] = xar;
    vec4<TE> acc[NB];
#pragma unroll
    for (int J = 0; J < NB; ++J) acc[J] = vec4<TE>{0, 0, 0, 0};
#pragma unroll
    for (int p = 0; p < Q / 2; ++p) {
      asm volatile("" ::: "memory");  // the reads of later pairs stay below
      TE2 A[NB];
#pragma unroll
      for (int J = 0; J < NB; ++J) A[J] = *reinterpret_cast<const TE2*>(lt + 16 * J * LD + 8 * p);
#pragma unroll
      for (int J = 0; J < NB; ++J) acc[J] = mfma(A[J].x, b[2 * p], acc[J]);
#pragma unroll
      for (int J = 0; J < NB; ++J) acc[J] = mfma(A[J].y, b[2 * p + 1], acc[J]);
    }
#pragma unroll
    for (int J = 0; J < NB; ++J)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int col = 16 * J + drow<TE>(kk, r);
        if (rok && col < N) Out[row + (int64_t)col * ldO] = out_value<MODE, TE>(acc[J][r], xar, infl);
      }
  }
}

// 65 <= N <= 128: R = M^-1/2 (FP32 for FP32 members) from ymat, 32 rows at a time
// through LDS in two buffers - the whole would leave one workgroup a CU with its
// loads, products and stores one after another - while each of eight waves keeps
// a strip of 16 rows; the next rows are in flight during a product, and the
// four waves on a SIMD belong to two workgroups.  The product is with R; row k of T
// is row k of R plus p_k + q_k v (OmegaRow, in slots 0 and 3 of vec), so a row of
// Sf adds its products with p and q; row N - 1 in ymat is that of T^T already.
// 64 800 zones of 121 rows, N = 128: 7.2 ms FP64 (26.9 GB moved: 3.7 TB/s), 4.2 FP32
// (13.6 GB; T whole in LDS, and a pass for the mean: 9.3 + 1.35 and 4.85 + 0.7).  Omega on
// the way to LDS cost 0.7 to 1.2 ms more, in k_func's registers 3.4 ms of spills there.
template <int MODE, typename TE>
__global__ __launch_bounds__(512, 4) void k_update128(int64_t z0, const int32_t* __restrict__ zorder, int N,
                                                      const int64_t* __restrict__ sel_ptr,
                                                      const int64_t* __restrict__ zone_ptr,
                                                      const double* __restrict__ ymat,
                                                      const double* __restrict__ vec,
                                                      const double* __restrict__ X0,
                                                      const TE* __restrict__ S, int64_t ldS,
                                                      double* __restrict__ xa, TE* __restrict__ Out,
                                                      int64_t ldO, double scaling, double infl,
                                                      double maxcorr,
                                                      const double* __restrict__ maxcorr_v) {
  constexpr int NP = 128, Q = NP / 4, CB = 32, LD = sizeof(TE) == 4 ? NP + 4 : NP + 2;
  typedef TE TE2 __attribute__((ext_vector_type(2)));
  typedef TE TEV __attribute__((ext_vector_type(16 / sizeof(TE))));
  constexpr int EV = 16 / sizeof(TE), NV = 4 / EV;  // 16-byte pieces of a thread's 4 entries
  __shared__ __attribute__((aligned(16))) TE L[2][CB * LD];
  __shared__ __attribute__((aligned(16))) double as[NP], p[NP], q[NP], v[NP];
  const int zl = blockIdx.x;
  const int64_t z = zone_at(zorder, z0 + zl);
  const int64_t i0 = zone_ptr[z], sz = zone_ptr[z + 1] - i0;
  if (sz <= 0) return;
  const int tid = threadIdx.x;
  const bool active = sel_ptr[z + 1] > sel_ptr[z];  // else T = I, a = 0
  const TE* X = reinterpret_cast<const TE*>(ymat + (size_t)zl * NP * NP);
  const double* Vz = vec + (size_t)zl * 4 * NP;
  if (tid < NP) {
    const double a = Vz[NP + tid];
    as[tid] = MODE == 1 ? a / scaling : a;
    p[tid] = active ? Vz[tid] : 0.0;
    q[tid] = active ? Vz[3 * NP + tid] : 0.0;
    v[tid] = active ? Vz[2 * NP + tid] : 0.0;
  }
  // thread t moves entries 4 (t % 16) .. + 3 of each half of row t / 16 of a
  // block, a half at a time: with both in registers beside the strip, the FP64
  // kernel spilled (34 GB moved instead of 27, 8.4 ms)
  TEV st[NV];
  auto fetch = [&](int h, int t, int half) {
    const int sr = t >> 4, sc = 4 * (t & 15) + 64 * half;
#pragma unroll
    for (int w = 0; w < NV; ++w)
      st[w] = *reinterpret_cast<const TEV*>(X + (size_t)(CB * h + sr) * NP + sc + EV * w);
    if (!active)
#pragma unroll
      for (int w = 0; w < NV; ++w)
#pragma unroll
        for (int i = 0; i < EV; ++i) st[w][i] = CB * h + sr == sc + EV * w + i ? (TE)1 : (TE)0;
  };
  auto put = [&](int h, int t, int half) {
    const int sr = t >> 4, sc = 4 * (t & 15) + 64 * half;
#pragma unroll
    for (int w = 0; w < NV; ++w)
      *reinterpret_cast<TEV*>(L[h & 1] + sr * LD + sc + EV * w) = st[w];
  };
  const int nh = (N + CB - 1) / CB;
  for (int64_t r0 = 0; r0 < sz; r0 += 128) {
    // the thread index opaque in each pass: loads, addresses and predicates made
    // from it would else be formed ahead of the loop, and spill
    int tp = threadIdx.x;
    asm volatile("" : "+v"(tp));
    const int wave = __builtin_amdgcn_readfirstlane(tp >> 6), li = tp & 15, kk = (tp >> 4) & 3;
    auto k_of = [&](int q) { return 8 * (q >> 1) + 2 * kk + (q & 1); };
    const int64_t rb = r0 + 16 * wave;
    const bool rok = rb + li < sz;
    const int64_t row = i0 + (rok ? rb + li : 0);
    TE b[Q];
    fetch(0, tp, 0);
    if (rb < sz) load_members(b, S, row, ldS, kk, N);
    put(0, tp, 0);
    fetch(0, tp, 1);
    put(0, tp, 1);
    lds_barrier();
    double xar = 0.0, gp = 0.0, gq = 0.0;
    if (rb < sz) {
      xar = strip_head<Q, MODE>(b, N, k_of, [&](int q) { return as[k_of(q)]; }, rok, row, X0, maxcorr,
                                maxcorr_v);
      if (MODE == 0 && rok && kk == 0) xa[row] = xar;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        if (i % 4 == 0) asm volatile("" ::: "memory");  // the vectors piece by piece
        gp = fma((double)b[i], p[k_of(i)], gp);
        gq = fma((double)b[i], q[k_of(i)], gq);
      }
      gp = sum_xor32(sum_xor16(gp));
      gq = sum_xor32(sum_xor16(gq));
      opaque(b);
    }
#pragma unroll 1
    for (int h = 0; h < nh; ++h) {
      int tq = threadIdx.x;
      asm volatile("" : "+v"(tq));
      const int li = tq & 15, kk = (tq >> 4) & 3;
      if (h + 1 < nh) fetch(h + 1, tq, 0);
      const TE* lt = L[h & 1] + li * LD + 2 * kk;
      vec4<TE> acc[2] = {};
      auto product = [&](int half) {
#pragma unroll
        for (int e = 0; e < Q / 4; ++e) {
          const int g = half * (Q / 4) + e;
          asm volatile("" ::: "memory");  // the reads of later pairs stay below
          TE2 A[2];
#pragma unroll
          for (int J = 0; J < 2; ++J) A[J] = *reinterpret_cast<const TE2*>(lt + 16 * J * LD + 8 * g);
#pragma unroll
          for (int J = 0; J < 2; ++J) acc[J] = mfma(A[J].x, b[2 * g], acc[J]);
#pragma unroll
          for (int J = 0; J < 2; ++J) acc[J] = mfma(A[J].y, b[2 * g + 1], acc[J]);
        }
      };
      if (rb < sz) product(0);
      if (h + 1 < nh) {
        put(h + 1, tq, 0);
        fetch(h + 1, tq, 1);
      }
      if (rb < sz) {
        product(1);
#pragma unroll
        for (int J = 0; J < 2; ++J)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int col = CB * h + 16 * J + drow<TE>(kk, r);
            const double y = (double)acc[J][r] + (col < N - 1 ? fma(gq, v[col], gp) : 0.0);
            if (rok && col < N) Out[row + (int64_t)col * ldO] = out_value<MODE, TE>(y, xar, infl);
          }
      }
      if (h + 1 < nh) put(h + 1, tq, 1);
      lds_barrier();
    }
  }
}

// Waves per zone at N <= 32: one for every 32 rows of a mean zone, at most
// the four of a workgroup (a wave reads the whole of T).
void launch_update(int NP, const ChunkArgs& A, hipStream_t st) {
  const int wpz = A.zone_rows > 64 ? 4 : (A.zone_rows > 32 ? 2 : 1);
  const dim3 small((unsigned)(((int64_t)A.nzc * wpz + 3) / 4)), blk(256);
#define OAK_UPD(MODE, TE, SRC, DST)                                                                   \
  switch (NP) {                                                                                       \
    case 16:                                                                                          \
      hipLaunchKernelGGL((k_update_small<16, MODE, TE>), small, blk, 0, st, A.z0, A.zorder, A.nzc, wpz, \
                         A.N, A.zone_ptr, A.mat, A.vec, A.X0, SRC, A.ldS, A.xa, DST, A.ldO, A.scaling, \
                         A.infl, A.maxcorr, A.maxcorr_v);                                             \
      break;                                                                                          \
    case 32:                                                                                          \
      hipLaunchKernelGGL((k_update_small<32, MODE, TE>), small, blk, 0, st, A.z0, A.zorder, A.nzc, wpz, \
                         A.N, A.zone_ptr, A.mat, A.vec, A.X0, SRC, A.ldS, A.xa, DST, A.ldO, A.scaling, \
                         A.infl, A.maxcorr, A.maxcorr_v);                                             \
      break;                                                                                          \
    case 64:                                                                                          \
      if (A.N <= 48)                                                                                  \
        hipLaunchKernelGGL((k_update64<MODE, TE, 3>), dim3(A.nzc), blk, 0, st, A.z0, A.zorder, A.N,   \
                           A.sel_ptr, A.zone_ptr, A.ymat, A.vec, A.X0, SRC, A.ldS, A.xa, DST, A.ldO,  \
                           A.scaling, A.infl, A.maxcorr, A.maxcorr_v);                                \
      else                                                                                            \
        hipLaunchKernelGGL((k_update64<MODE, TE, 4>), dim3(A.nzc), blk, 0, st, A.z0, A.zorder, A.N,   \
                           A.sel_ptr, A.zone_ptr, A.ymat, A.vec, A.X0, SRC, A.ldS, A.xa, DST, A.ldO,  \
                           A.scaling, A.infl, A.maxcorr, A.maxcorr_v);                                \
      break;                                                                                          \
    case 128:                                                                                         \
      hipLaunchKernelGGL((k_update128<MODE, TE>), dim3(A.nzc), dim3(512), 0, st, A.z0, A.zorder, A.N, \
                         A.sel_ptr, A.zone_ptr, A.ymat, A.vec, A.X0, SRC, A.ldS, A.xa, DST, A.ldO,    \
                         A.scaling, A.infl, A.maxcorr, A.maxcorr_v);                                  \
      break;                                                                                          \
  }
  if (A.prec == 1) {
    OAK_UPD(1, float, A.S32, A.Out32)
  } else if (A.mode == 0) {
    OAK_UPD(0, double, A.S, A.Out)
  } else {
    OAK_UPD(1, double, A.S, A.Out)
  }
#undef OAK_UPD
}

}  // namespace oakg
