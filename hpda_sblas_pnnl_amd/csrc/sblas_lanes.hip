// sblas_lanes.hip -- row blocks whose rows are summed by groups of lanes, x in
// FP64, for gfx950: the measure behind the x precision of narrow values.
//
// Whether FP32 / BF16 values in row blocks gather x from an FP32 copy decides
// what a caller gets (a normwise error of about 2e-8 or of 1e-15), so it must not
// follow the speed of the kernels that multiply: those change.  A plan's trial
// times this kernel beside the others and takes the copy where it is not slower
// than the column-sorted form (Plan::choose_csr); no product runs it.  Its loads,
// LDS (28 KB at 8 elements a thread, five workgroups a CU) and lane groups are
// therefore kept as they are, whatever the row blocks of row_block_device.hpp
// become.  What bounds it: five workgroups a CU against their eight, and lanes
// that wait for their wave's longest row.  us, this kernel / those / column-sorted,
// FP32 values: banded 625,057 rows of 13 28.5 / 25.5 / 29.3, 793,650 rows of 28
// 66 / 58 / 63; R-MAT 117,821 rows 22.5 / 14.3 / 18.6.
#include "internal.hpp"
#include "row_block_device.hpp"
#include "rows_device.hpp"

namespace sblas {
namespace {

// One row block per workgroup.  Phase 1 issues every global load the block
// needs that does not depend on another: ITEMS values and columns per thread,
// the block's row pointers and, with beta != 0, its y entries; then the x
// gathers.  Row pointers go to LDS and y stays in registers, so the row sums
// (phase 2, SUBW lanes per row, products read from LDS) and the y writes (phase
// 3, consecutive threads on consecutive rows) wait on no further memory round
// trip.  A block that holds a piece of one long row sums in registers and
// reduces across the whole workgroup instead.
template <typename VT, int ITEMS, int SUBW>
__global__ __launch_bounds__(kStreamBlock) void k_csr_lanes(
    const RowBlock *__restrict__ blocks, int nblocks, int xcd_remap,
    const int *__restrict__ rp, const int *__restrict__ col, const VT *__restrict__ val,
    const double *__restrict__ x, double *__restrict__ y, double alpha, double beta,
    double *__restrict__ partials) {
  constexpr int BLOCK = kStreamBlock;
  constexpr int CAP = BLOCK * ITEMS;
  constexpr int RPT = (kStreamRowsMax + BLOCK) / BLOCK;  // row pointers per thread
  constexpr int YPT = kStreamRowsMax / BLOCK;            // rows per thread in phase 3
  __shared__ double prod[CAP];
  __shared__ double ysh[kStreamRowsMax];
  __shared__ int rps[kStreamRowsMax + 1];
  __shared__ double wsum[BLOCK / 64];
  const int b = rows::logical_block(nblocks, xcd_remap);
  if (b < 0) return;
  const RowBlock rb = blocks[b];
  const int lo = rb.lo, hi = rb.hi;
  const int t = threadIdx.x;
  const int r0 = rb.row_begin, nrows = rb.row_end - rb.row_begin;

  // phase 1.  Lanes past the window re-read its last element and their product
  // is dropped by a select; row pointer and y addresses are clamped into the
  // block's rows, so no load sits under a branch.
  double p[ITEMS];
  // the first row's bounds, the same for every thread (the long-row test
  // below must be uniform over the workgroup)
  const int rp_first = rp[r0], rp_second = rp[r0 + 1];
  int rpv[RPT];
#pragma unroll
  for (int k = 0; k < RPT; k++) rpv[k] = rp[r0 + min(t + k * BLOCK, nrows)];
  double yv[YPT];
  if (beta != 0.0) {
#pragma unroll
    for (int k = 0; k < YPT; k++) yv[k] = y[r0 + min(t + k * BLOCK, nrows - 1)];
  } else {
#pragma unroll
    for (int k = 0; k < YPT; k++) yv[k] = 0.0;
  }
  if (hi > lo) {
    double v[ITEMS];
    int c[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) {
      const int e = min(lo + t + k * BLOCK, hi - 1);
      v[k] = rows::load_val(val, e);
      c[k] = rows::load_col(col, e);
    }
    double xv[ITEMS];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) xv[k] = x[c[k]];
#pragma unroll
    for (int k = 0; k < ITEMS; k++) p[k] = (lo + t + k * BLOCK < hi) ? v[k] * xv[k] : 0.0;
  } else {
#pragma unroll
    for (int k = 0; k < ITEMS; k++) p[k] = 0.0;
  }

  if (nrows == 1 && (rp_first < lo || rp_second > hi)) {
    // piece of a long row: register sum, wave reduction, then across waves
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < ITEMS; k++) s += p[k];
    s = rows::lanes_sum<64>(s);
    if ((t & 63) == 0) wsum[t >> 6] = s;
    __syncthreads();
    if (t == 0) {
      double total = 0.0;
#pragma unroll
      for (int w = 0; w < BLOCK / 64; w++) total += wsum[w];
      partials[2 * b] = total;
    }
    return;
  }
#pragma unroll
  for (int k = 0; k < ITEMS; k++) {
    const int e = t + k * BLOCK;
    if (e < hi - lo) prod[e] = p[k];
  }
#pragma unroll
  for (int k = 0; k < RPT; k++)
    if (t + k * BLOCK <= nrows) rps[t + k * BLOCK] = rpv[k];
  __syncthreads();

  // phase 2: one group of SUBW lanes per row, whole waves for long rows
  rows::block_row_sums<SUBW, BLOCK>(prod, rps, nrows, lo, hi, ysh);
  __syncthreads();

  // phase 3: y for whole rows, partials for rows cut by the window
#pragma unroll
  for (int k = 0; k < YPT; k++) {
    const int i = t + k * BLOCK;
    if (i < nrows) {
      const double s = ysh[i];
      if ((i == 0 || i == nrows - 1) && (rps[i] < lo || rps[i + 1] > hi)) {
        partials[2 * b + (i == 0 ? 0 : 1)] = s;
      } else {
        y[r0 + i] = (beta == 0.0) ? alpha * s : alpha * s + beta * yv[k];
      }
    }
  }
}

template <typename VT, int ITEMS>
int lanes_items(const StreamLaunch &L, const RowBlock *blocks, const int *rp, const int *col,
                const VT *val, const double *x, double *y, double alpha, double beta,
                double *partials, hipStream_t s) {
  const dim3 grid(L.grid), block(kStreamBlock);
#define SBLAS_LANES_CASE(W)                                                                     \
  case W:                                                                                       \
    hipLaunchKernelGGL((k_csr_lanes<VT, ITEMS, W>), grid, block, 0, s, blocks, L.nblocks,       \
                       L.xcd_remap, rp, col, val, x, y, alpha, beta, partials);                 \
    break;
  switch (L.subwave) {
    SBLAS_LANES_CASE(1)
    SBLAS_LANES_CASE(2)
    SBLAS_LANES_CASE(4)
    SBLAS_LANES_CASE(8)
    SBLAS_LANES_CASE(16)
    SBLAS_LANES_CASE(32)
    SBLAS_LANES_CASE(64)
    default:
      set_error(SBLAS_ERR_ARGS, "lane groups: lanes per row must be a power of two in [1, 64]");
      return SBLAS_ERR_ARGS;
  }
#undef SBLAS_LANES_CASE
  SBLAS_HIP_TRY(hipGetLastError());
  return SBLAS_OK;
}

template <typename VT>
int lanes_typed(const StreamLaunch &L, const RowBlock *blocks, const int *rp, const int *col,
                const VT *val, const double *x, double *y, double alpha, double beta,
                double *partials, hipStream_t s) {
  return L.items == 16
             ? lanes_items<VT, 16>(L, blocks, rp, col, val, x, y, alpha, beta, partials, s)
             : lanes_items<VT, 8>(L, blocks, rp, col, val, x, y, alpha, beta, partials, s);
}

}  // namespace

int launch_csr_lanes(int val_type, const StreamLaunch &L, const RowBlock *blocks, const int *rp,
                     const int *col, const void *val, const double *x, double *y, double alpha,
                     double beta, double *partials, hipStream_t s) {
  if (L.grid <= 0) return SBLAS_OK;
  if (L.items != 8 && L.items != 16) {
    set_error(SBLAS_ERR_ARGS, "lane groups: items per thread must be 8 or 16");
    return SBLAS_ERR_ARGS;
  }
  switch (val_type) {
    case SBLAS_VAL_F32:
      return lanes_typed(L, blocks, rp, col, static_cast<const float *>(val), x, y, alpha, beta,
                         partials, s);
    case SBLAS_VAL_BF16:
      return lanes_typed(L, blocks, rp, col, static_cast<const uint16_t *>(val), x, y, alpha, beta,
                         partials, s);
    default:
      set_error(SBLAS_ERR_ARGS, "lane groups: FP32 or BF16 values");
      return SBLAS_ERR_ARGS;
  }
}

}  // namespace sblas
