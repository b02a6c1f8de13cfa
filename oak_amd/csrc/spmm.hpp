// The observation operator on the members, shared by the FP64 and FP32 states.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"
#include "spmm_grid.hpp"

namespace oakg {

// HEc[l + k m] = Hshift[l] + sum_e val_e E[col_e, k] over the entries e of row
// l, in their order (FP64 members: rounded after each product and sum, as
// OAK's loop; FP32 members: fused).
//
// Bound by the lines of E that the gathers touch.  Workgroups go to the XCDs
// in turn, so workgroup b takes members b % 8, b % 8 + 8, ...: each member's
// lines enter one XCD's L2 instead of all eight.  A thread takes kSpmmMembers
// of them, which reads the row's indices once for all, and four entries at a
// time, so that 16 gathers are in flight.  201 000 rows of 4 entries, 100 FP32
// members: 0.85 ms with a member per grid row and one entry at a time, 0.55 so.
// (grid: spmm_grid)
template <typename TE>
__global__ __launch_bounds__(256) void k_spmm_obs(int64_t m, int64_t n, int N,
                                                  const int64_t* __restrict__ row_ptr,
                                                  const int32_t* __restrict__ col,
                                                  const double* __restrict__ val,
                                                  const TE* __restrict__ E, int64_t ld,
                                                  const TE* __restrict__ Hshift,
                                                  double* __restrict__ HEc,
                                                  unsigned* __restrict__ err) {
#pragma clang fp contract(off)
  constexpr int MB = kSpmmMembers;
  const int k0 = spmm_member(blockIdx.x, blockIdx.y);
  const int64_t l = spmm_row(blockIdx.x, blockIdx.z) + threadIdx.x;
  if (k0 >= N || l >= m) return;
  const TE* Ek[MB];
#pragma unroll
  for (int q = 0; q < MB; ++q) Ek[q] = E + (int64_t)(k0 + 8 * q < N ? k0 + 8 * q : k0) * ld;
  double s[MB];
#pragma unroll
  for (int q = 0; q < MB; ++q) s[q] = 0;
  const int64_t e0 = row_ptr[l], e1 = row_ptr[l + 1];
  bool bad = n <= 0 && e0 < e1;
  for (int64_t e = e0; e < e1 && n > 0; e += 4) {
    double v[4];
    TE x[4][MB];
    bool take[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t ec = e + u < e1 ? e + u : e1 - 1;
      const int32_t j = col[ec];
      v[u] = val[ec];
      const bool in = j >= 0 && j < n;
      bad = bad || !in;
      take[u] = in && e + u < e1;
#pragma unroll
      for (int q = 0; q < MB; ++q) x[u][q] = Ek[q][in ? j : 0];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int q = 0; q < MB; ++q) {
        double t;
        if (sizeof(TE) == 8) {
          t = v[u] * (double)x[u][q];
          t = s[q] + t;
        } else {
          t = fma(v[u], (double)x[u][q], s[q]);
        }
        s[q] = take[u] ? t : s[q];
      }
  }
  if (bad) atomicOr(err, OAKG_DERR_IDX);
  const double h = (double)Hshift[l];
#pragma unroll
  for (int q = 0; q < MB; ++q)
    if (k0 + 8 * q < N) HEc[l + (int64_t)(k0 + 8 * q) * m] = s[q] + h;
}

}  // namespace oakg
