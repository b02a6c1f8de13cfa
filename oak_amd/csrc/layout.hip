// State layout on the GPU: the zone permutation of ensembles when they are
// loaded and saved (loadVector/loadEnsemble and saveVector with
// ModML%permute, assimilation.F90:869-880, 901, 1268-1359): rows gathered
// from the full (land and sea) field vectors into the permuted sea-only
// state, and scattered back.
// A workgroup takes a run of kRows rows for its members: the indices are read
// once for all of them, eight elements a thread are in flight, and what the
// run touches of a field is read or written as whole lines by one L2,
// neighbouring runs being given to the same XCD (workgroups go to the eight
// XCDs in turn).  Where the state holds columns, the next row is a level away
// in the field and each lane of a wave would move its own line: with several
// members the run's indices are sorted first (once), and the elements pass
// through LDS between the state's order and the field's.
// HBM-bound.  5.25 million rows of 32 FP64 members, two thirds of the points
// sea at random (2.7 GB and the land in the lines), gathered and scattered: a
// row and member per thread 1.02 and 1.45 ms; runs 0.91 and 1.50; sorted
// 0.75 and 1.26 (a line written in part is read as well).
#include <stdint.h>

#include <algorithm>

#include "common.hpp"
#include "internal.hpp"

namespace oakg {

constexpr int kRows = 2048, kPer = kRows / 256;

template <typename T, bool GATHER, bool SORT>
__global__ __launch_bounds__(256) void k_permute_rows(int64_t n, int N, int members, unsigned nx,
                                                      const int64_t* __restrict__ idx,
                                                      const T* __restrict__ in, int64_t ldi,
                                                      T* __restrict__ out, int64_t ldo,
                                                      int64_t lim, unsigned* __restrict__ err) {
  __shared__ union {
    uint64_t key[SORT ? kRows : 1];
    T buf[2][SORT ? kRows : 1];
  } S;
  const unsigned per = gridDim.x / 8, run = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (run >= nx) return;
  const int t = threadIdx.x;
  const int64_t l0 = (int64_t)run * kRows + t;
  int64_t j[kPer];
  bool ok[kPer], bad = false;
#pragma unroll
  for (int i = 0; i < kPer; ++i) j[i] = idx[l0 + 256 * i < n ? l0 + 256 * i : n - 1];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const bool in_range = j[i] >= 0 && j[i] < lim;
    bad = bad || !in_range;
    ok[i] = in_range && l0 + 256 * i < n;
    j[i] = in_range ? j[i] : 0;
  }
  if (bad && blockIdx.y == 0) atomicOr(err, OAKG_DERR_IDX);
  if (lim <= 0) return;
  const int ka = blockIdx.y * members, kb = min(N, ka + members);
  if (SORT) {
    // the place in the run, in the low bits, goes along (and ends up in loc);
    // rows not to be moved sort to the end
    int loc[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      S.key[256 * i + t] = ok[i] ? ((uint64_t)j[i] * kRows | (unsigned)(256 * i + t)) : ~0ull;
    for (int size = 2; size <= kRows; size *= 2)
      for (int d = size / 2; d > 0; d /= 2) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kPer / 2; ++i) {
          const int p = 256 * i + t, a = 2 * p - (p & (d - 1)), b = a + d;
          const uint64_t x = S.key[a], y = S.key[b];
          if ((x > y) == ((a & size) == 0)) {
            S.key[a] = y;
            S.key[b] = x;
          }
        }
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const uint64_t x = S.key[256 * i + t];
      const bool moves = x != ~0ull;
      j[i] = moves ? (int64_t)(x / kRows) : 0;
      loc[i] = moves ? (int)(x & (kRows - 1)) : -1;
    }
    __syncthreads();
    T v[kPer];
    auto load = [&](int k) {
      const T* ik = in + (int64_t)k * ldi;
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        v[i] = ik[GATHER ? j[i] : (l0 + 256 * i < n ? l0 + 256 * i : n - 1)];
    };
    load(ka);
    for (int k = ka; k < kb; ++k) {
      T* okp = out + (int64_t)k * ldo;
      T* buf = S.buf[k & 1];
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        if (!GATHER)
          buf[256 * i + t] = v[i];
        else if (loc[i] >= 0)
          buf[loc[i]] = v[i];
      }
      lds_barrier();
      if (k + 1 < kb) load(k + 1);
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        if (GATHER) {
          if (ok[i]) okp[l0 + 256 * i] = buf[256 * i + t];
        } else {
          if (loc[i] >= 0) okp[j[i]] = buf[loc[i]];
        }
      }
    }
    return;
  }
  for (int k = ka; k < kb; ++k) {
    const T* ik = in + (int64_t)k * ldi;
    T* okp = out + (int64_t)k * ldo;
    T v[kPer];
    // every load in range, also those not stored, so that none waits for another
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      v[i] = ik[GATHER ? j[i] : (l0 + 256 * i < n ? l0 + 256 * i : n - 1)];
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      if (ok[i]) okp[GATHER ? l0 + 256 * i : j[i]] = v[i];
  }
}

// All members in a workgroup when the runs alone fill the device (16
// workgroups a CU), else in as many groups as bring it there.
void launch_permute_rows(bool gather, int elem, int64_t n, int N, const int64_t* idx,
                         const void* in, int64_t ldi, void* out, int64_t ldo, int64_t lim,
                         unsigned* err, hipStream_t st) {
  if (n <= 0 || N <= 0) return;
  const unsigned nx = (unsigned)((n + kRows - 1) / kRows), gx = (nx + 7) / 8 * 8;
  const int groups = (int)std::min<int64_t>(N, std::max<int64_t>(1, (4096 + gx - 1) / gx));
  const int members = (N + groups - 1) / groups;
  const dim3 grid(gx, (unsigned)((N + members - 1) / members)), blk(256);
  // the sort pays from eight members a workgroup on: gathered and scattered, 31
  // and 46 us a member without it, 34 and 46 with it at four, 25 and 42 at eight
  // (indices past 2^52 have no room for it)
  const bool sort = members >= 8 && lim < ((int64_t)1 << 52);
#define OAK_PERMUTE_S(T, G, SRT)                                                                   \
  hipLaunchKernelGGL((k_permute_rows<T, G, SRT>), grid, blk, 0, st, n, N, members, nx, idx,        \
                     (const T*)in, ldi, (T*)out, ldo, lim, err)
#define OAK_PERMUTE(T, G)          \
  if (sort)                        \
    OAK_PERMUTE_S(T, G, true);     \
  else                             \
    OAK_PERMUTE_S(T, G, false)
  if (elem == 8) {
    if (gather) {
      OAK_PERMUTE(double, true);
    } else {
      OAK_PERMUTE(double, false);
    }
  } else {
    if (gather) {
      OAK_PERMUTE(float, true);
    } else {
      OAK_PERMUTE(float, false);
    }
  }
#undef OAK_PERMUTE_S
#undef OAK_PERMUTE
}

}  // namespace oakg
