// Observation operator from coordinates (interp.hip): grid, search levels
// and launch interfaces.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace oakg {

// A model variable's grid on the device: n dims, nodes per dim, node
// coordinates per dim (first index fastest), the mask (1 = land) and the
// node -> state column map (-1: not in the state; NULL: the node index).
struct GridDev {
  int n;
  int64_t shape[4];
  const double* coord[4];
  const uint8_t* mask;
  const int64_t* state;
};

// The search tree's levels (interp.hip): level k < depth holds the bounds of
// its boxes from offset off[k] on, 2 n doubles a box (minima, then maxima).
struct BoxLevels {
  int depth;        // levels that are stored (the cells below are not)
  int dim_depth[4]; // splits after which every interval of the dim is one cell
  int32_t cells[4];
  int64_t off[32];
  int64_t total;    // boxes of all levels
};

struct ObsPosDev {
  const int32_t* var;
  const double *x, *y, *z, *t;
};

int tet_count(int n);
std::vector<double> tet_table(int n);
BoxLevels box_levels(int n, const int64_t* shape);

void launch_obs_interp(int n, int64_t m, int var, const GridDev& g,
                       const BoxLevels& bl, double* bounds, const double* tc, int nbth, const ObsPosDev& o, int slot_stride,
                       int32_t* slot_col, double* slot_w, int64_t* counts, uint8_t* valid,
                       unsigned* status, hipStream_t st);
void launch_obs_compact(int64_t m, int slot_stride, const int64_t* row_ptr,
                        const int32_t* slot_col, const double* slot_w, int32_t* col, double* val,
                        hipStream_t st);

}  // namespace oakg
