// Observation operator from coordinates on the GPU: genObservationOper
// (assimilation.F90:2471-2656) with cinterp (ndgrid.F90:1183-1257), the
// databox search of ndgrid_inc.F90:534-990 and the hyper-tetrahedral
// interpolation of ndgrid.F90:357-665, followed by packSparseMatrix
// (assimilation.F90:4132-4208) and the zone permutation of the state columns
// (assimilation.F90:2404-2409).
//
// One thread per observation: a depth-first walk of the grid's box tree, the
// cell test of the candidate leaves (InCube: the first simplex of the cell's
// split that holds the point) with the 2^n corner weights of the cell.  The
// tree is never stored as one: its boxes follow from the grid's shape, and
// only the bounds of the boxes above the cells are computed, on the device.  The arithmetic of the
// simplex test and weights runs in the same order as the host restatement
// (sums in index order, LU with partial pivoting, no contraction), so
// indices and weights are reproducible bit for bit.
#include <math.h>
#include <string.h>

#include <algorithm>
#include <vector>

#include "common.hpp"
#include "interp.hpp"

namespace oakg {

constexpr double kTetTol = 1e-8;  // interp_tetrahedron, ndgrid.F90:474

static int factorial_i(int n) {
  int f = 1;
  for (int i = 2; i <= n; ++i) f *= i;
  return f;
}

int tet_count(int n) { return factorial_i(n) * (1 << (n - 1)); }

// split (ndgrid.F90:357-435) into the slab starting at simplex l0 of the
// column-major table tc(2^n, n+1, nbth): entry (j, k, l) at j + 2^n (k + (n+1) l).
static void split_tab(int n, int subn, const int* fixeddim, const int* sel, double* tc, int l0) {
  const int twon = 1 << n, ldk = twon, ldl = twon * (n + 1);
  if (subn == 1) {
    for (int k = 0; k < 2; ++k)
      for (int j = 0; j < twon; ++j) tc[j + ldk * k + ldl * l0] = 0.0;
    int k = 0;
    for (int j = 0; j < twon; ++j)
      if (sel[j]) tc[j + ldk * (k++) + ldl * l0] = 1.0;
    return;
  }
  int cnt = 0;
  for (int j = 0; j < twon; ++j) cnt += sel[j] != 0;
  const int nb = factorial_i(subn) * (1 << (subn - 1));
  const int sub_nb = factorial_i(subn - 1) * (1 << (subn - 2));
  for (int l = 0; l < nb; ++l)
    for (int j = 0; j < twon; ++j) tc[j + ldk * subn + ldl * (l0 + l)] = sel[j] ? 1.0 / cnt : 0.0;
  int m = 0;
  for (int i = 0; i < n; ++i) {
    if (fixeddim[i]) continue;
    int fd[4] = {0, 0, 0, 0}, sub[16];
    for (int d = 0; d < n; ++d) fd[d] = fixeddim[d];
    fd[i] = 1;
    for (int side = 0; side <= 1; ++side) {
      for (int k = 0; k < twon; ++k) sub[k] = sel[k] && (((k >> i) & 1) == side);
      split_tab(n, subn - 1, fd, sub, tc, l0 + m);
      m += sub_nb;
    }
  }
}

std::vector<double> tet_table(int n) {
  std::vector<double> tc((size_t)(1 << n) * (n + 1) * tet_count(n), 0.0);
  int fixed[4] = {0, 0, 0, 0}, sel[16];
  for (int j = 0; j < (1 << n); ++j) sel[j] = 1;
  split_tab(n, n, fixed, sel, tc.data(), 0);
  return tc;
}

// The box tree of locate_databox: a box is a range of node indices per dim; a
// box with a side above 1 is split in every dim at im = (imin + imax) / 2 (bit
// d of the child's number set: [imin, im], else [im, imax]); a box with no
// side above 1 is a cell.  A side of 1 gives itself and then the point
// [imin, imin], a point itself twice, so that a tree over a grid whose sides
// differ holds each cell many times (2^(n depth) boxes; built and uploaded by
// the host, 2 million boxes and 290 ms for 120 x 90 x 20 nodes; the whole call
// with the levels below: 1.1 ms).
//
// Only the order of the cells in the walk and each cell's own bounds decide
// the result: a box's bounds hold its cells' bounds, so tests above the cells
// only prune.  A box with a point in some dim comes after the box that has the
// side itself in its place and whose cells, with wider bounds, include its
// own: it gives no hit that the walk has not had.  So the walk splits only the
// sides above 1, and level k has per dim the 2^k intervals of level k, or the
// cells once every interval is one.
BoxLevels box_levels(int n, const int64_t* shape) {
  BoxLevels b{};
  for (int d = 0; d < n; ++d) {
    b.cells[d] = (int32_t)(shape[d] - 1);
    while (((int64_t)1 << b.dim_depth[d]) < b.cells[d]) ++b.dim_depth[d];
    b.depth = std::max(b.depth, b.dim_depth[d]);
  }
  for (int k = 0; k < b.depth; ++k) {
    int64_t c = 1;
    for (int d = 0; d < n; ++d) c *= k < b.dim_depth[d] ? (int64_t)1 << k : b.cells[d];
    b.off[k] = b.total;
    b.total += c;
  }
  return b;
}

// ---------------------------------------------------------------------------
// Device side
// ---------------------------------------------------------------------------
// Barycentric coordinates c of xi in the simplex X (n x (n+1), column-major)
// (interp_tetrahedron, ndgrid.F90:464-629, non-degenerate branch).  Returns
// 0 inside, 1 outside, 2 degenerate (|det| <= tol).
template <int N>
__device__ int tet_coeff(const double* X, const double* xi, double* c) {
#pragma clang fp contract(off)
  constexpr int M = N + 1;
  double A[M][M], b[M], xc[N];
#pragma unroll
  for (int d = 0; d < N; ++d) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < M; ++k) s = s + X[d + N * k];
    xc[d] = s / M;
  }
#pragma unroll
  for (int k = 0; k < M; ++k) A[0][k] = 1.0;
#pragma unroll
  for (int d = 0; d < N; ++d)
#pragma unroll
    for (int k = 0; k < M; ++k) A[d + 1][k] = X[d + N * k] - xc[d];
  b[0] = 1.0;
#pragma unroll
  for (int d = 0; d < N; ++d) b[d + 1] = xi[d] - xc[d];
  double det = 1.0;
  bool zero_piv = false;
#pragma unroll
  for (int j = 0; j < M; ++j) {
    if (zero_piv) break;
    int p = j;
    double best = fabs(A[j][j]);
#pragma unroll
    for (int i = j + 1; i < M; ++i)
      if (fabs(A[i][j]) > best) {
        best = fabs(A[i][j]);
        p = i;
      }
    if (p != j) {
#pragma unroll
      for (int i = j + 1; i < M; ++i)
        if (i == p) {
#pragma unroll
          for (int k = 0; k < M; ++k) {
            const double t = A[j][k];
            A[j][k] = A[i][k];
            A[i][k] = t;
          }
          const double t = b[j];
          b[j] = b[i];
          b[i] = t;
        }
      det = -det;
    }
    const double piv = A[j][j];
    det = det * piv;
    if (piv == 0.0) {
      zero_piv = true;
      continue;
    }
#pragma unroll
    for (int i = j + 1; i < M; ++i) {
      const double l = A[i][j] / piv;
#pragma unroll
      for (int k = j + 1; k < M; ++k) A[i][k] = A[i][k] - l * A[j][k];
      b[i] = b[i] - l * b[j];
    }
  }
  if (!(fabs(det) > kTetTol)) return 2;
#pragma unroll
  for (int i = M - 1; i >= 0; --i) {
    double s = b[i];
#pragma unroll
    for (int k = i + 1; k < M; ++k) s = s - A[i][k] * c[k];
    c[i] = s / A[i][i];
  }
  int out = 0;
#pragma unroll
  for (int k = 0; k < M; ++k)
    if (!(0.0 - kTetTol <= c[k] && c[k] <= 1.0 + kTetTol)) out = 1;
  return out;
}

// interp_cube (ndgrid.F90:636-665): the first simplex of the split holding
// xi; its 2^n corner weights into w (if not null).  0 inside, 1 outside,
// 2 degenerate.
template <int N>
__device__ int cube_coeff(const double* __restrict__ tc, int nbth, const double* px,
                          const double* xi, double* w) {
#pragma clang fp contract(off)
  constexpr int TWON = 1 << N, M = N + 1;
  for (int l = 0; l < nbth; ++l) {
    const double* t = tc + (size_t)TWON * M * l;
    double X[N * M], c[M];
#pragma unroll
    for (int d = 0; d < N; ++d)
#pragma unroll
      for (int k = 0; k < M; ++k) {
        double s = 0.0;
#pragma unroll
        for (int j = 0; j < TWON; ++j) s = s + px[d + N * j] * t[j + TWON * k];
        X[d + N * k] = s;
      }
    const int r = tet_coeff<N>(X, xi, c);
    if (r == 2) return 2;
    if (r == 0) {
      if (w) {
#pragma unroll
        for (int j = 0; j < TWON; ++j) {
          double s = 0.0;
#pragma unroll
          for (int k = 0; k < M; ++k) s = s + t[j + TWON * k] * c[k];
          w[j] = s;
        }
      }
      return 0;
    }
  }
  return 1;
}

// Corner points of the cell with lower corner ind; corner j takes index
// min(ind + 1, shape - 1) along the set bits of j (InCube); node indices out.
template <int N>
__device__ void cell_corners(const GridDev& g, const int32_t* ind, double* px, int64_t* node) {
  constexpr int TWON = 1 << N;
#pragma unroll
  for (int j = 0; j < TWON; ++j) {
    int64_t l = 0, off = 1;
#pragma unroll
    for (int d = 0; d < N; ++d) {
      int64_t p = ind[d];
      if ((j >> d) & 1) p = ind[d] + 1 < g.shape[d] - 1 ? ind[d] + 1 : g.shape[d] - 1;
      l += p * off;
      off *= g.shape[d];
    }
    if (node) node[j] = l;
#pragma unroll
    for (int d = 0; d < N; ++d) px[d + N * j] = g.coord[d][l];
  }
}

// The interval [lo, hi] with number id of a dim at level k (all intervals are
// one cell after kd splits): its child `bit` one level down; an interval of
// one cell has itself (bit 0).  Numbers count a level's intervals, from kd on
// the cells.
__device__ __forceinline__ void child_interval(int k, int kd, int bit, int32_t& lo, int32_t& hi,
                                               int32_t& id) {
  const int32_t im = lo + (hi - lo) / 2;
  if (bit)
    hi = im;
  else
    lo = im;
  id = k + 1 < kd ? 2 * id + 1 - bit : lo;
}

// Bounds of the boxes of level k: from the nodes (the lowest level, sides of
// at most 2) or from the level below.  Comparisons that fail for NaN leave it
// out.  One thread per box; a grid of 120 x 90 x 20 nodes has 1e5 boxes in all.
template <int N, bool NODES>
__global__ __launch_bounds__(256) void k_box_bounds(GridDev g, BoxLevels bl, int k, int64_t count,
                                                    double* __restrict__ bounds) {
  constexpr int TWON = 1 << N;
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= count) return;
  double mn[N], mx[N];
#pragma unroll
  for (int d = 0; d < N; ++d) {
    mn[d] = HUGE_VAL;
    mx[d] = -HUGE_VAL;
  }
  int64_t r = b;
  int32_t lo[N], hi[N], id[N];
#pragma unroll
  for (int d = 0; d < N; ++d) {
    const int kd = bl.dim_depth[d];
    const int64_t c = k < kd ? (int64_t)1 << k : bl.cells[d];
    id[d] = (int32_t)(r % c);
    r /= c;
    if (k < kd) {
      lo[d] = 0;
      hi[d] = bl.cells[d];
      for (int i = k - 1; i >= 0; --i) {
        const int32_t im = lo[d] + (hi[d] - lo[d]) / 2;
        if ((id[d] >> i) & 1)
          lo[d] = im;
        else
          hi[d] = im;
      }
    } else {
      lo[d] = id[d];
      hi[d] = id[d] + 1;
    }
  }
  if (NODES) {
    int32_t p[N];
#pragma unroll
    for (int d = 0; d < N; ++d) p[d] = lo[d];
    for (;;) {
      int64_t l = 0, off = 1;
#pragma unroll
      for (int d = 0; d < N; ++d) {
        l += p[d] * off;
        off *= g.shape[d];
      }
#pragma unroll
      for (int d = 0; d < N; ++d) {
        const double x = g.coord[d][l];
        if (x < mn[d]) mn[d] = x;
        if (x > mx[d]) mx[d] = x;
      }
      bool more = false;
#pragma unroll
      for (int d = 0; d < N; ++d)
        if (!more) {
          if (p[d] < hi[d]) {
            ++p[d];
            more = true;
          } else {
            p[d] = lo[d];
          }
        }
      if (!more) break;
    }
  } else {
#pragma unroll
    for (int q = 0; q < TWON; ++q) {
      int64_t l = 0, off = 1;
#pragma unroll
      for (int d = 0; d < N; ++d) {
        const int kd = bl.dim_depth[d];
        int32_t clo = lo[d], chi = hi[d], cid = id[d];
        child_interval(k, kd, hi[d] - lo[d] > 1 ? (q >> d) & 1 : 0, clo, chi, cid);
        l += cid * off;
        off *= k + 1 < kd ? (int64_t)1 << (k + 1) : bl.cells[d];
      }
      const double* c = bounds + 2 * N * (bl.off[k + 1] + l);
#pragma unroll
      for (int d = 0; d < N; ++d) {
        if (c[d] < mn[d]) mn[d] = c[d];
        if (c[N + d] > mx[d]) mx[d] = c[N + d];
      }
    }
  }
  double* o = bounds + 2 * N * (bl.off[k] + b);
#pragma unroll
  for (int d = 0; d < N; ++d) {
    o[d] = mn[d];
    o[N + d] = mx[d];
  }
}

// Pass 1: per observation of variable var, the cell (depth-first search of
// the box tree), the corner weights, and the entries of its row of H in the
// slots [stride l, stride l + 2^n): state column (or -1: no entry) and
// weight (the slots of every observation start out as -1).
// counts[l] = number of entries, valid[l] = validobs, status bit 1 for a
// degenerate cell (OAKG_EUNSUP).
//
// Bound by latency (one chain of dependent loads and divisions per thread), so
// waves of one workgroup each, and the bounds of a box's 2^n children are
// loaded together: the walk keeps, per level, the children still to visit as
// a mask, and rebuilds a box from the masks when it comes back to it.
template <int N>
__global__ __launch_bounds__(64) void k_obs_interp(int64_t m, int var, GridDev g, BoxLevels bl,
                                                   const double* __restrict__ bounds,
                                                   const double* __restrict__ tc, int nbth,
                                                   const int32_t* __restrict__ obs_var,
                                                   const double* __restrict__ ox,
                                                   const double* __restrict__ oy,
                                                   const double* __restrict__ oz,
                                                   const double* __restrict__ ot, int stride,
                                                   int32_t* __restrict__ slot_col,
                                                   double* __restrict__ slot_w,
                                                   int64_t* __restrict__ counts,
                                                   uint8_t* __restrict__ valid,
                                                   unsigned* __restrict__ status) {
  constexpr int TWON = 1 << N;
  const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= m) return;
  if (obs_var[l] != var) return;
  double xi[N];
  const double* oc[4] = {ox, oy, oz, ot};
#pragma unroll
  for (int d = 0; d < N; ++d) xi[d] = oc[d][l];
  bool hit = false;
  int64_t node[TWON];
  double w[TWON];
  // the cell with lower corner lo.  0: holds xi (its nodes and weights are
  // set), 1: does not, 2: degenerate
  auto test_cell = [&](const int32_t* lo) -> int {
    double px[N * TWON];
    cell_corners<N>(g, lo, px, node);
    bool in = true;
#pragma unroll
    for (int d = 0; d < N; ++d) {
      double mn = HUGE_VAL, mx = -HUGE_VAL;
#pragma unroll
      for (int j = 0; j < TWON; ++j) {
        const double x = px[d + N * j];
        if (x < mn) mn = x;
        if (x > mx) mx = x;
      }
      in = in && !(xi[d] < mn || xi[d] > mx);
    }
    return in ? cube_coeff<N>(tc, nbth, px, xi, w) : 1;
  };
  // the box of the walk at level k and the mask of its children to visit
  uint16_t todo[32];
  int32_t lo[N], hi[N], id[N];
  int k = 0;
  auto to_root = [&]() {
#pragma unroll
    for (int d = 0; d < N; ++d) {
      lo[d] = 0;
      hi[d] = bl.cells[d];
      id[d] = bl.dim_depth[d] > 0 ? 0 : lo[d];
    }
  };
  auto children = [&]() -> unsigned {
    unsigned mask = 0;
#pragma unroll
    for (int q = 0; q < TWON; ++q) {
      bool leaf = true, copy = false;
      int64_t at = 0, off = 1;
#pragma unroll
      for (int d = 0; d < N; ++d) {
        const int kd = bl.dim_depth[d], bit = (q >> d) & 1;
        copy = copy || (bit && hi[d] - lo[d] <= 1);
        int32_t a = lo[d], b = hi[d], c = id[d];
        child_interval(k, kd, bit, a, b, c);
        leaf = leaf && b - a <= 1;
        at += c * off;
        off *= k + 1 < kd ? (int64_t)1 << (k + 1) : bl.cells[d];
      }
      bool in = true;
      if (!leaf) {
        const double* c = bounds + 2 * N * (bl.off[k + 1] + at);
#pragma unroll
        for (int d = 0; d < N; ++d) in = in && !(xi[d] < c[d] || xi[d] > c[N + d]);
      }
      mask |= (unsigned)(in && !copy) << q;
    }
    return mask;
  };
  to_root();
  if (bl.depth == 0) {
    const int r = test_cell(lo);
    if (r == 2) atomicOr(status, 1u);
    hit = r == 0;
  } else {
    bool in = true;
#pragma unroll
    for (int d = 0; d < N; ++d) in = in && !(xi[d] < bounds[d] || xi[d] > bounds[N + d]);
    todo[0] = in ? children() : 0;
    for (;;) {
      if (todo[k] == 0) {
        // back to the box above, rebuilt from the children taken
        if (k == 0) break;
        const int up = k - 1;
        to_root();
        for (k = 0; k < up; ++k) {
          const int q = __ffs(todo[k]) - 1;
#pragma unroll
          for (int d = 0; d < N; ++d)
            child_interval(k, bl.dim_depth[d], (q >> d) & 1, lo[d], hi[d], id[d]);
        }
        todo[k] &= todo[k] - 1;
        continue;
      }
      const int q = __ffs(todo[k]) - 1;
      int32_t a[N], b[N], c[N];
      bool leaf = true;
#pragma unroll
      for (int d = 0; d < N; ++d) {
        a[d] = lo[d];
        b[d] = hi[d];
        c[d] = id[d];
        child_interval(k, bl.dim_depth[d], (q >> d) & 1, a[d], b[d], c[d]);
        leaf = leaf && b[d] - a[d] <= 1;
      }
      if (leaf) {
        const int r = test_cell(a);
        if (r == 2) atomicOr(status, 1u);
        hit = r == 0;
        if (r != 1) break;
        todo[k] &= todo[k] - 1;
      } else {
#pragma unroll
        for (int d = 0; d < N; ++d) {
          lo[d] = a[d];
          hi[d] = b[d];
          id[d] = c[d];
        }
        ++k;
        todo[k] = children();
      }
    }
  }
  int64_t cnt = 0;
  uint8_t ok = 0;
  if (hit) {
    // cinterp: masked corners put the point out of the grid
    bool masked = false;
    if (g.mask)
#pragma unroll
      for (int j = 0; j < TWON; ++j) masked = masked || g.mask[node[j]] != 0;
    // packSparseMatrix: entries of nodes outside the state are dropped;
    // validobs is the validity of the observation's last entry
    if (!masked)
#pragma unroll
      for (int j = 0; j < TWON; ++j) {
        const int64_t s = g.state ? g.state[node[j]] : node[j];
        slot_col[l * stride + j] = s >= 0 ? (int32_t)s : -1;
        slot_w[l * stride + j] = w[j];
        cnt += s >= 0;
        ok = s >= 0;
      }
  }
  if (!(hit && cnt > 0)) {
#pragma unroll
    for (int j = 0; j < TWON; ++j) slot_col[l * stride + j] = -1;
  }
  counts[l] = cnt;
  valid[l] = ok;
}

// Pass 2: compaction of the slots into CSR rows.
__global__ void k_obs_compact(int64_t m, int stride, const int64_t* __restrict__ row_ptr,
                              const int32_t* __restrict__ slot_col,
                              const double* __restrict__ slot_w, int32_t* __restrict__ col,
                              double* __restrict__ val) {
  const int64_t l = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= m) return;
  int64_t p = row_ptr[l];
  for (int j = 0; j < stride; ++j) {
    const int32_t s = slot_col[l * stride + j];
    if (s >= 0) {
      col[p] = s;
      val[p] = slot_w[l * stride + j];
      ++p;
    }
  }
}

template <int N>
static void obs_interp_t(int64_t m, int var, const GridDev& g, const BoxLevels& bl, double* bounds,
                         const double* tc, int nbth, const ObsPosDev& o, int slot_stride,
                         int32_t* slot_col, double* slot_w, int64_t* counts, uint8_t* valid,
                         unsigned* status, hipStream_t st) {
  for (int k = bl.depth - 1; k >= 0; --k) {
    const int64_t c = (k + 1 < bl.depth ? bl.off[k + 1] : bl.total) - bl.off[k];
    const dim3 grid((unsigned)((c + 255) / 256)), blk(256);
    if (k == bl.depth - 1)
      hipLaunchKernelGGL((k_box_bounds<N, true>), grid, blk, 0, st, g, bl, k, c, bounds);
    else
      hipLaunchKernelGGL((k_box_bounds<N, false>), grid, blk, 0, st, g, bl, k, c, bounds);
  }
  hipLaunchKernelGGL(k_obs_interp<N>, dim3((unsigned)((m + 63) / 64)), dim3(64), 0, st, m, var, g,
                     bl, bounds, tc, nbth, o.var, o.x, o.y, o.z, o.t, slot_stride, slot_col, slot_w,
                     counts, valid, status);
}

// Computes the grid's bounds into `bounds` (2 n bl.total doubles), then one
// pass over the observations.
void launch_obs_interp(int n, int64_t m, int var, const GridDev& g, const BoxLevels& bl,
                       double* bounds, const double* tc, int nbth, const ObsPosDev& o,
                       int slot_stride, int32_t* slot_col, double* slot_w, int64_t* counts,
                       uint8_t* valid, unsigned* status, hipStream_t st) {
#define OAK_INTERP(NN)                                                                           \
  obs_interp_t<NN>(m, var, g, bl, bounds, tc, nbth, o, slot_stride, slot_col, slot_w, counts,    \
                   valid, status, st)
  switch (n) {
    case 1: OAK_INTERP(1); break;
    case 2: OAK_INTERP(2); break;
    case 3: OAK_INTERP(3); break;
    case 4: OAK_INTERP(4); break;
  }
#undef OAK_INTERP
}

void launch_obs_compact(int64_t m, int slot_stride, const int64_t* row_ptr,
                        const int32_t* slot_col, const double* slot_w, int32_t* col, double* val,
                        hipStream_t st) {
  if (m > 0)
    hipLaunchKernelGGL(k_obs_compact, dim3((unsigned)((m + 255) / 256)), dim3(256), 0, st, m,
                       slot_stride, row_ptr, slot_col, slot_w, col, val);
}

}  // namespace oakg
