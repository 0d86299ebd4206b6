// row_block_device.hpp -- one row block of a CSR matrix by one workgroup, the
// body of the row-block kernel (sblas_vector.hip) and of the batch's row-block
// items (sblas_batch.hip).
#pragma once

#include "internal.hpp"
#include "span_device.hpp"

namespace sblas {
namespace rows {

// Stored value or column, streamed past the caches that hold x.
__device__ __forceinline__ double load_val(const double *p, int j) {
  return __builtin_nontemporal_load(p + j);
}
__device__ __forceinline__ double load_val(const float *p, int j) {
  return static_cast<double>(__builtin_nontemporal_load(p + j));
}
__device__ __forceinline__ double load_val(const uint16_t *p, int j) {
  const uint32_t h = __builtin_nontemporal_load(p + j);
  return static_cast<double>(__uint_as_float(h << 16));
}
__device__ __forceinline__ int load_col(const int *p, int j) {
  return __builtin_nontemporal_load(p + j);
}

// One row block by one workgroup.  Phase 1 issues every global load the block needs that does not
// depend on another: ITEMS values and columns per thread (consecutive threads
// on consecutive elements, so each load instruction of a wave covers whole
// cache lines), the bounds of the thread's rows and, with beta != 0, their y;
// then the x gathers, whose products go to LDS.  Phase 2 sums the rows by
// spans of elements (span_device.hpp).  Phase 3 writes y, consecutive threads
// on consecutive rows, from bounds that are still in registers.  XT float: x
// gathered from its FP32 copy (narrow values: half the bytes per gather and per
// cached line of x; an FP32 value times an FP32 x is exact in FP64, so x's
// rounding is the only one added).
//
// What bounds it: the x gathers, one L2 request an element (about 2.1e11 a
// second on this GPU), and on small matrices the chain of dependent loads.
// Against the form that gave each row a group of lanes, with the sums in an
// LDS array of their own (28 KB of LDS, 5 workgroups a CU; now 18.7 KB and 8),
// us before -> now, FP64: power law 20,000 rows 8.0 -> 6.9, 200,000 rows 25.5
// -> 22.3; R-MAT 30,000 rows 14.2 -> 10.1, 300,000 rows 38.6 -> 31.5, scale 22
// over column segments 463 -> 442; banded 100,000 rows of 140 56.6 -> 42.7.
//
// with_beta: beta != 0, y is read.  slots: two partial slots, for the block's
// first and last row where the window cuts them.  The body may be called again
// by the same workgroup without a barrier between.
template <typename VT, int ITEMS, typename XT>
__device__ __forceinline__ void row_block(const RowBlock &rb, bool with_beta,
                                          const int *__restrict__ rp, const int *__restrict__ col,
                                          const VT *__restrict__ val, const XT *__restrict__ x,
                                          double *__restrict__ y, double alpha, double beta,
                                          double *__restrict__ slots, span::Shared<ITEMS> &sh) {
  constexpr int B = span::kBlock;
  constexpr int RPT = kStreamRowsMax / B;  // rows per thread
  const int lo = rb.lo, hi = rb.hi;
  const int t = threadIdx.x;
  const int r0 = rb.row_begin, nrows = rb.row_end - rb.row_begin;
  span::clear_ends(sh);

  // phase 1.  Threads past the window re-read its last element (same cache
  // line), so no load sits under a divergent branch.
  double v[ITEMS];
  int c[ITEMS];
  if (hi > lo) {
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
      const int e = min(lo + t + k * B, hi - 1);
      v[k] = load_val(val, e);
      c[k] = load_col(col, e);
    }
  }
  int rs[RPT], re[RPT];
  double yv[RPT];
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    if (k == 0 || k * B < nrows) {
      const int r = r0 + min(t + k * B, nrows - 1);
      rs[k] = rp[r];
      re[k] = rp[r + 1];
      if (with_beta) yv[k] = y[r];
    }
  }
  __syncthreads();
  if (hi > lo) {
    XT xv[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) xv[k] = x[c[k]];
#pragma unroll
    for (int k = 0; k < RPT; k++)
      if (t + k * B < nrows && min(re[k], hi) > max(rs[k], lo))
        span::mark_end(sh, min(re[k], hi) - 1 - lo);
#pragma unroll
    for (int k = 0; k < ITEMS; k++)
      sh.prod[span::pos<ITEMS>(t + k * B)] = v[k] * static_cast<double>(xv[k]);
  }
  __syncthreads();

  // phase 2
  span::row_sums(sh);

  // phase 3: y for whole rows, partials for rows cut by the window
#pragma unroll
  for (int k = 0; k < RPT; k++) {
    const int i = t + k * B;
    if (i < nrows) {
      const int e = min(re[k], hi);
      const double s = e > max(rs[k], lo) ? sh.prod[span::pos<ITEMS>(e - 1 - lo)] : 0.0;
      if ((i == 0 || i == nrows - 1) && (rs[k] < lo || re[k] > hi)) {
        slots[i == 0 ? 0 : 1] = s;
      } else {
        y[r0 + i] = with_beta ? alpha * s + beta * yv[k] : alpha * s;
      }
    }
  }
}

}  // namespace rows
}  // namespace sblas
