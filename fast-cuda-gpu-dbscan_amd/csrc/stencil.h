// Device helpers shared by the clustering kernels and the one-step
// baseline: coordinate loads, the FP64 neighbour predicate, and the point
// ranges of a cell's rows.
#pragma once
#include "internal.h"

namespace dclust {

// ------------------------------------------------------------ predicates --
// FP64 coordinates of cell-sorted point i.  The FP32 form keeps no sorted
// FP64 copy (only its guard-band rechecks need FP64): they are read from
// the caller's rows.
template <int D, bool F32>
__device__ __forceinline__ void load_x(const Dev& d, int32_t i, double* x) {
  if constexpr (F32) {
    const double* p = d.xrow[i];
#pragma unroll
    for (int k = 0; k < D; ++k) x[k] = p[k];
  } else {
#pragma unroll
    for (int k = 0; k < D; ++k) x[k] = d.X[3 * (int64_t)i + k];
  }
}
template <int D>
__device__ __forceinline__ void load_g(const Dev& d, int32_t i, uint32_t* g) {
#pragma unroll
  for (int k = 0; k < D; ++k) g[k] = d.G[3 * (int64_t)i + k];
}

// fl(fl(fl(d0^2) + fl(d1^2)) [+ fl(d2^2)]), left to right
template <int D>
__device__ __forceinline__ double d2_64(const double* a, const double* b) {
  double t = a[0] - b[0];
  double s = t * t;
#pragma unroll
  for (int k = 1; k < D; ++k) {
    double u = a[k] - b[k];
    double v = u * u;
    s = s + v;
  }
  return s;
}

// the oracle's box of a range query centred on c: fl(c-eps) <= q <= fl(c+eps)
template <int D>
__device__ __forceinline__ bool box_64(const double* c, const double* q, double eps) {
  bool in = true;
#pragma unroll
  for (int k = 0; k < D; ++k) {
    const double lo = c[k] - eps, hi = c[k] + eps;
    in = in && lo <= q[k] && q[k] <= hi;
  }
  return in;
}

// points of a row's cells (consecutive): [a, e)
__device__ __forceinline__ void row_points(const Dev& d, uint2 row, int32_t& a, int32_t& e) {
  a = e = 0;
  if (row.y) {
    a = d.cell_start[row.x];
    e = d.cell_start[row.x + row_cells(row)];
  }
}

}  // namespace dclust
