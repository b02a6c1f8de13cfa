// The launch of k_spmm_obs: which rows and members a workgroup takes.
#pragma once
#include <stdint.h>

namespace oakg {

constexpr int kSpmmMembers = 4;                    // of a thread, 8 apart
constexpr int64_t kSpmmRowBlocks = (int64_t)1 << 20;  // of 256 rows along x

// Along x the 8 workgroups of a block of 256 rows, one for each XCD, along y the groups
// of 8 kSpmmMembers members.  8 threads a row along one dimension reach the 2^32 threads
// of a launch at 2^29 rows (with the groups in it as well: at 2^29 rows over their
// number); more rows go along z.
struct SpmmGrid {
  unsigned x, y, z;
};
inline SpmmGrid spmm_grid(int64_t m, int N) {
  const int64_t nb = (m + 255) / 256, nx = nb < kSpmmRowBlocks ? nb : kSpmmRowBlocks;
  return {(unsigned)(8 * nx), (unsigned)((N + 8 * kSpmmMembers - 1) / (8 * kSpmmMembers)),
          (unsigned)((nb + nx - 1) / nx)};
}
// of workgroup (bx, by, bz): its first row; its first member
constexpr int64_t spmm_row(unsigned bx, unsigned bz) {
  return 256 * (kSpmmRowBlocks * (int64_t)bz + (bx >> 3));
}
constexpr int spmm_member(unsigned bx, unsigned by) { return (int)(8 * kSpmmMembers * by + (bx & 7)); }

}  // namespace oakg
